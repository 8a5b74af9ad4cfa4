// tpm_pp.hip -- fused short-range PP + mesh interpolation + kick.
//
// Reference: kick_treepm_kernel (kick_treepm.cu:460-759) and kick_pme_kernel
// (kick_pme.cu:128-357).  Work item here = one tile of <= TS active
// sinks of one chain cell (tpm_tiles.hip), processed by one wave64: lane l holds sink
// l % TS and walks source stream l / TS (64 / TS streams over one shared
// source list), the streams are summed at the end.
//
// Source staging: the wave walks the 27 neighbour cells (the candidate set
// of kick_pme.cu:265-318) 64 particles at a time; each lane tests one source
// against the box of the tile's active sinks and survivors are compacted
// (ballot + mbcnt) into LDS, as exact int32 offsets (near sources) or float
// offsets (far ones) from the box's centre.  A source whose box
// distance exceeds rcut has r >= rcut to every sink, so dropping it changes
// no result; smaller tiles have tighter boxes and drop more.  Near pairs
// evaluate compute_pp_interaction (kick_treepm.cu:242-283), far ones the same
// law without its softening (pp_far).  kick_pme evaluates every pair with the former
// (pp_sum_pme).
//
// Near pairs: distances are int32(sink - source) converted to float, which is the
// reference's distance() (gravity_short.hpp:20-22) in units of 2^-32; every
// constant is pre-scaled by the matching power of two so the FP32 arithmetic
// is the reference's up to exact power-of-two factors, except that inside
// the softening length the two (erfc - 1) corrections are evaluated by their
// series in x^2 (pp_law), where the formula as written cancels to nothing in
// FP32.  The self pair is
// evaluated like any other source, as in the reference: inside the
// softening branch it contributes -35/16 h^-1 to phi and nothing to g.
#include <algorithm>
#include <cmath>
#include <type_traits>
#include <vector>

#include "tpm_pp_device.hpp"
#include "tpm_tiles.hpp"

#include <climits>

// Staged sources of a wave: far ones (float offsets) and near ones (int32
// offsets), 5 KiB of LDS together, so 32 waves fill a CU's 160 KiB.  A list
// is flushed when a further round of 64 might not fit.
#define FAR_AT 112
#define FAR_CAP 208   // FAR_AT + 64 + 32: four rounds of padding for 8 streams
#define NEAR_AT 48
#define NEAR_CAP 112  // NEAR_AT + 64
// Per-sink source lists (LISTS, 16-sink tiles): a flush of <= LCAP staged
// sources (staging flushes above LFLUSH), the far dummy at LFAR.
#define LCAP 144
#define LFLUSH (LCAP - 64)
#define LSBUF 160
#define LFAR (LSBUF - 1)

// Every fused multiply-add in this file is written out (fmaf) and the
// compiler may fuse nothing else, so the results come out the same bits in
// every instantiation of the kernel (single box, batch, persistent).
#pragma clang fp contract(off)

namespace {

struct PPArgs {
    const uint32_t* __restrict__ x;
    const uint32_t* __restrict__ y;
    const uint32_t* __restrict__ z;
    float* __restrict__ vx;
    float* __restrict__ vy;
    float* __restrict__ vz;
    int8_t* __restrict__ rung;
    float* __restrict__ gx;
    float* __restrict__ gy;
    float* __restrict__ gz;
    float* __restrict__ pot;
    const int32_t* __restrict__ cell_begin;
    const int4* __restrict__ tiles;
    const int32_t* __restrict__ ntiles;
    const uint32_t* __restrict__ order;  // the particles of a tile: order[tile.y .. tile.z)
    const float4* __restrict__ mesh;  // mesh force and potential per sink, made before the launch
                                      // by mesh_force_kernel (nullptr: no mesh term)
    unsigned long long* __restrict__ counters;
    int* __restrict__ queue;        // 8 per-XCD tile queues (persistent launch)
    const tpm_box_dev* __restrict__ boxes;  // batched: per-box table, tile.w = box
    tpm_box_dev box0;                        // single box
    unsigned flags;
};

// The fused kernel.  Work item = one tile: TS sinks of one chain cell
// against the culled sources of the 27 neighbour cells, then mesh
// interpolation and the kick epilogue.
//   PERSIST = false: one workgroup per tile.  The hardware deals workgroups
//     round-robin over the 8 XCDs, so each XCD gets one contiguous
//     (spatially coherent) run of tiles and its L2 keeps the shared
//     neighbour cells.
//   PERSIST = true: resident workgroups take tiles from 8 queues, one
//     contiguous run per XCD; a workgroup drains its own XCD's queue first
//     and then helps the others.  Every queue ends, so every workgroup exits.
// BATCH = true: tile.w names the box whose constants apply (device table).
// PME = true: kick_pme's pair law (the caller turns culling and phi0 off).
// The box record of a tile.  A batch's table is read word by word through
// the constant address space, so the record arrives by scalar loads in SGPRs
// (the table is not written during the launch); read as ordinary global
// memory, its fields would take vector registers.
template <bool BATCH>
__device__ __forceinline__ tpm_box_dev tile_box(const PPArgs& a, int w) {
    if constexpr (BATCH) {
        static_assert(sizeof(tpm_box_dev) % 4 == 0, "box record of whole words");
        constexpr int NW = (int)(sizeof(tpm_box_dev) / 4);
        using cword = const __attribute__((address_space(4))) int;
        cword* src = (cword*)(a.boxes + __builtin_amdgcn_readfirstlane(w));
        int words[NW];
#pragma unroll
        for (int k = 0; k < NW; k++) words[k] = src[k];
        tpm_box_dev b;
        __builtin_memcpy(&b, words, sizeof b);
        return b;
    } else {
        return a.box0;
    }
}

// The same record, read through the argument block la (the launch's PPArgs).
template <bool BATCH>
__device__ __forceinline__ tpm_box_dev late_box(const __attribute__((address_space(4))) PPArgs* la, int w) {
    constexpr int NW = (int)(sizeof(tpm_box_dev) / 4);
    using cword = const __attribute__((address_space(4))) int;
    cword* src;
    if constexpr (BATCH)
        src = (cword*)(la->boxes + __builtin_amdgcn_readfirstlane(w));
    else
        src = (cword*)&la->box0;
    int words[NW];
#pragma unroll
    for (int k = 0; k < NW; k++) words[k] = src[k];
    tpm_box_dev b;
    __builtin_memcpy(&b, words, sizeof b);
    return b;
}

// f(integral_constant<int, k>) for k = 0 .. N-1, k a constant expression
// in each call.
template <int K, int N>
struct static_for_t {
    template <class F>
    static __device__ __forceinline__ void run(F& f) {
        f(std::integral_constant<int, K>{});
        static_for_t<K + 1, N>::run(f);
    }
};
template <int N>
struct static_for_t<N, N> {
    template <class F>
    static __device__ __forceinline__ void run(F&) {}
};
template <int N, class F>
__device__ __forceinline__ void static_for(F& f) {
    static_for_t<0, N>::run(f);
}

// Minimum / maximum over the TS sinks of a tile (every stream holds a copy of
// them): the 16-lane steps are DPP moves, the wider ones shuffles.
template <int TS, class Op>
__device__ __forceinline__ int tile_reduce(int v, Op op) {
    v = op(v, __builtin_amdgcn_update_dpp(v, v, 0xB1, 0xf, 0xf, false));   // lane ^ 1
    v = op(v, __builtin_amdgcn_update_dpp(v, v, 0x4E, 0xf, 0xf, false));   // lane ^ 2
    v = op(v, __builtin_amdgcn_update_dpp(v, v, 0x141, 0xf, 0xf, false));  // half-row mirror: the other four
    if constexpr (TS > 8) v = op(v, __builtin_amdgcn_update_dpp(v, v, 0x140, 0xf, 0xf, false));  // row mirror
#pragma unroll
    for (int o = 16; o < TS; o <<= 1) v = op(v, __shfl_xor(v, o));
    return v;
}
template <int TS>
__device__ __forceinline__ int tile_min(int v) {
    return tile_reduce<TS>(v, [](int a, int b) { return min(a, b); });
}
template <int TS>
__device__ __forceinline__ int tile_max(int v) {
    return tile_reduce<TS>(v, [](int a, int b) { return max(a, b); });
}

// The short-range sums of one tile, by one wave: lane l has sink l % TS (raw
// position px, py, pz) and walks stream l / TS.  The sources are those of the
// 27 cells around cell (cx, cy, cz), 64 at a time, as int32 offsets from the
// centre of the tile's box, rounded to float once (2^-24 of the offset, which
// is at most the pair's distance and half the box).  Each source is tested
// against that box:
//   beyond the cutoff (far_cull2, a margin of 2048 raw units over rcut, float
//     rounding stays below 600): dropped.  The offset f of a source is the
//     nearest image's, |f| <= 2^31, so on each axis every sink of the box is at least
//     |f| - the half width away, round the box too (C < 5);
//   within far_near2 of the box: near list, as int32 offsets, evaluated with
//     the general law (pp_pair);
//   else: far list, as float offsets, evaluated with pp_far.  Every pair of a
//     far source is at least FAR_X0 2 rs and h apart.
// At 512^3 nine pairs of ten are far ones.
// The float offsets' rounding grows with the box's half width H: a pair at
// distance d is off by up to 2^-23 (d + H) per axis, where an exact difference
// is rounded by 2^-24 d.  H is 1.1 rs in a full cell and at most 2.5 rs in the
// sparsest at the usual ratios (half a cell); a wider box (few sinks in a
// chain mesh much coarser than rcut) keeps the exact integer differences: its
// sources all take the near list.  Error of a sink's pair sum against FP64
// relative to the rms force, median over the sinks, exact differences and the
// general law for every pair / this: 64^3 particles C = 11 1.9e-7 / 1.4e-7,
// C = 5 2.0e-7 / 1.5e-7, 93^3 C = 5 3.1e-7 / 2.3e-7, 128^3 C = 5 2.3e-7 / 1.8e-7,
// 20^3 on a 128^3 mesh, C = 5, 2.4e-8 for both.
// (Offsets from the cells' centres stored once per chain mesh save the
// conversions, but their rounding is that of a cell's width: 2.6e-7 at 128^3
// C = 5, and a close pair is off by 2e-6 in cells of 160 rs.  Kicks at the
// reference's ratios are 3 % slower without them, 120^3 25.6 -> 26.5 ms, the others the same.)
// The cutoff of a far pair: float offsets are rounded by up to a few raw
// units, and a pair on the wrong side of the cutoff is an error of
// 5e-4 of a typical force, larger than all rounding together.  So u is
// compared with both ends of a window that covers its rounding; a flush that
// met a pair inside the window (about one in 200 at 512^3) is followed by a
// pass that adds those of them whose exact squared integer offset is inside;
// near pairs that close to the cutoff are decided the same way (pp_pair_cut,
// pp_pair_open).  The decision is then the same for every tile size and
// order.
template <int TS, class Sync>
__device__ __forceinline__ void pp_sum(const PPArgs& a, const tpm_box_dev& B, int cx, int cy, int cz, uint32_t px,
                                       uint32_t py, uint32_t pz, uint32_t rx, uint32_t ry, uint32_t rz, bool inbox,
                                       int nact, float4* __restrict__ fbuf, int4* __restrict__ nbuf, Sync lds_sync,
                                       float& gx, float& gy, float& gz, float& ph, unsigned long long& executed) {
    constexpr int SPLIT = 64 / TS;  // source streams per wave
    constexpr int BLK = 4 * SPLIT;  // sources of a block of the far loop
    static_assert(TS >= 8 && FAR_AT + 64 + BLK <= FAR_CAP, "room for the padding");
    const int lane = (int)lane_id();
    const int stream = lane / TS;
    const int C = B.C;
    const bool cull = B.cull != 0;
    // the box of the sinks with inbox: centre (raw) and half widths
    int ox = (int)(px - rx), oy = (int)(py - ry), oz = (int)(pz - rz);
    const int lox = tile_min<TS>(inbox ? ox : INT_MAX), hix = tile_max<TS>(inbox ? ox : INT_MIN);
    const int loy = tile_min<TS>(inbox ? oy : INT_MAX), hiy = tile_max<TS>(inbox ? oy : INT_MIN);
    const int loz = tile_min<TS>(inbox ? oz : INT_MAX), hiz = tile_max<TS>(inbox ? oz : INT_MIN);
    // halves first: hi - lo may exceed 2^31 - 1 only for a cell wider than
    // half the box, which C >= 3 rules out, but lo + hi may not fit
    const int mx = lox + (hix - lox) / 2, my = loy + (hiy - loy) / 2, mz = loz + (hiz - loz) / 2;
    const uint32_t qx = rx + (uint32_t)mx, qy = ry + (uint32_t)my, qz = rz + (uint32_t)mz;
    const float hx = (float)max(hix - mx, mx - lox), hy = (float)max(hiy - my, my - loy),
                hz = (float)max(hiz - mz, mz - loz);
    const float near2 = fmaxf(hx, fmaxf(hy, hz)) > B.far_wide ? B.far_all2 : B.far_near2;
    // every pair of a near source is closer than rcut: no pair to decide
    const float reach = sqrtf(near2) + 2.f * sqrtf(fmaf(hx, hx, fmaf(hy, hy, hz * hz))) + 4096.f;
    const bool near_in = __builtin_amdgcn_readfirstlane(reach * reach < B.rcut2s);
    ox -= mx;
    oy -= my;
    oz -= mz;
    const float fox = (float)ox, foy = (float)oy, foz = (float)oz;
    // kept in vector registers: an SGPR operand costs a VALU instruction half its rate
    float ulo = B.far_ulo, uhi = B.far_uhi, fu = B.far_u;
    asm volatile("" : "+v"(ulo), "+v"(uhi), "+v"(fu));
    // lane l < 27: neighbour cell l's particles
    int rb = 0, re = 0;
    if (lane < 27) {
        int jx = cx + lane % 3 - 1, jy = cy + (lane / 3) % 3 - 1, jz = cz + lane / 9 - 1;
        jx += jx < 0 ? C : (jx >= C ? -C : 0);
        jy += jy < 0 ? C : (jy >= C ? -C : 0);
        jz += jz < 0 ? C : (jz >= C ? -C : 0);
        const int c2 = B.cell0 + (jz * C + jy) * C + jx;
        rb = a.cell_begin[c2];
        re = a.cell_begin[c2 + 1];
        // A cell out of reach of the box is left out as a whole.  Its
        // centre's offset ex, taken as the nearest image, puts a particle
        // of it at least |ex| - half a cell - the box's half width away on
        // that axis; a cell's planes are within C of k cell_w, 512 covers that.
        // (Cells of rcut keep nearly all 27.  Staging every candidate of
        // coarser ones cost more than the far law saved: chain mesh and kick
        // of 64^3 at C = 5 1.81 ms, now 1.11, 128^3 at C = 11 7.5, now 3.7.)
        const uint32_t w = B.cell_w;
        const float hw = (float)(w / 2) + 512.f;
        const float ex = fmaxf(fabsf((float)(int)((uint32_t)jx * w + w / 2 - qx)) - hw - hx, 0.f);
        const float ey = fmaxf(fabsf((float)(int)((uint32_t)jy * w + w / 2 - qy)) - hw - hy, 0.f);
        const float ez = fmaxf(fabsf((float)(int)((uint32_t)jz * w + w / 2 - qz)) - hw - hz, 0.f);
        if (fmaf(ex, ex, fmaf(ey, ey, ez * ez)) >= B.far_cull2) re = rb;
    }
    const uint32_t lane4 = 4u * (uint32_t)lane;
    gx = gy = gz = ph = 0.f;
    float ngx = 0.f, ngy = 0.f, ngz = 0.f, nph = 0.f;
    int nfar = 0, nnear = 0;
    int cell = -1, j0 = 0, je = 0;
    for (;;) {
        // 64 sources, or after the last cell none
        bool more = true;
        while (j0 >= je) {
            if (++cell == 27) {
                more = false;
                break;
            }
            j0 = __builtin_amdgcn_readlane(rb, cell);
            je = __builtin_amdgcn_readlane(re, cell);
        }
        if (more) {
            // lanes past the cell's end read its last particle and are masked
            const int left = je - j0;
            const unsigned long long valid = left >= 64 ? ~0ull : (1ull << left) - 1ull;
            const uint32_t off = min(lane4, 4u * (uint32_t)(left - 1));
            const int ix = (int)(*(const uint32_t*)((const char*)(a.x + j0) + off) - qx);
            const int iy = (int)(*(const uint32_t*)((const char*)(a.y + j0) + off) - qy);
            const int iz = (int)(*(const uint32_t*)((const char*)(a.z + j0) + off) - qz);
            const float fx = (float)ix, fy = (float)iy, fz = (float)iz;
            const float ex = fmaxf(fabsf(fx) - hx, 0.f), ey = fmaxf(fabsf(fy) - hy, 0.f),
                        ez = fmaxf(fabsf(fz) - hz, 0.f);
            const float d2 = fmaf(ex, ex, fmaf(ey, ey, ez * ez));
            unsigned long long mn = __ballot(d2 < near2), mf;
            mf = __ballot(d2 < B.far_cull2);
            if (!cull)
                // a difference of float offsets does not wrap round the
                // box as the int32 one does: sources for which it would
                // (C < 5) take the general law
                mn |= mf & __ballot(fmaxf(fabsf(fx) + hx, fmaxf(fabsf(fy) + hy, fabsf(fz) + hz)) > B.far_wrap);
            mf &= ~mn & valid;
            mn &= valid;
            const int j = j0 + lane;
            if (mf) {
                if (__builtin_amdgcn_inverse_ballot_w64(mf))
                    fbuf[__builtin_amdgcn_mbcnt_hi((unsigned)(mf >> 32),
                                                   __builtin_amdgcn_mbcnt_lo((unsigned)mf, nfar))] =
                        make_float4(fx, fy, fz, __int_as_float(j));
                nfar += __popcll(mf);
            }
            if (mn) {
                if (__builtin_amdgcn_inverse_ballot_w64(mn))
                    nbuf[__builtin_amdgcn_mbcnt_hi((unsigned)(mn >> 32),
                                                   __builtin_amdgcn_mbcnt_lo((unsigned)mn, nnear))] =
                        make_int4(ix, iy, iz, j);
                nnear += __popcll(mn);
            }
            j0 += 64;
        }
        if (nfar > FAR_AT || (!more && nfar > 0)) {
            // Whole blocks of 4 rounds (four pairs in flight per lane: 85
            // cycles per 64 pairs, some 12 more with two); the rest stays in the list,
            // and after the last source is filled up with padding sources
            // beyond any cutoff (e = 0).
            int nblk = nfar / BLK * BLK;
            if (!more && nblk < nfar) {
                if (lane < BLK) fbuf[nfar + lane] = make_float4(1e15f, 1e15f, 1e15f, 0.f);
                nblk += BLK;
            }
            lds_sync();
            unsigned long long window = 0ull;
#pragma unroll 1
            for (int q = 0; q < nblk; q += BLK) {
                float4 s[4];
#pragma unroll
                for (int k = 0; k < 4; k++) s[k] = fbuf[q + k * SPLIT + stream];
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    pp_far_cut(s[k], fox, foy, foz, fu, ulo, uhi, window, gx, gy, gz, ph);
                }
            }
            if (window) {
                for (int q = 0; q < nblk; q += SPLIT) {
                    const float4 s = fbuf[q + stream];
                    const float dx = s.x - fox, dy = s.y - foy, dz = s.z - foz;
                    const float u = fmaf(dx, dx, fmaf(dy, dy, dz * dz)) * fu;
                    if (u >= ulo && u < uhi) {
                        const int j = __float_as_int(s.w);
                        if (pp_inside(B, (int)((qx + (uint32_t)ox) - a.x[j]), (int)((qy + (uint32_t)oy) - a.y[j]),
                                      (int)((qz + (uint32_t)oz) - a.z[j])))
                            pp_far(dx, dy, dz, u, __builtin_amdgcn_exp2f(-u), gx, gy, gz, ph);
                    }
                }
            }
            const int done = min(nblk, nfar), rest = nfar - done;
            executed += (unsigned long long)done * (unsigned long long)nact;
            if (rest > 0) {
                const float4 t = fbuf[done + min(lane, rest - 1)];
                lds_sync();
                if (lane < rest) fbuf[lane] = t;
            }
            nfar = rest;
            lds_sync();
        }
        if (nnear > NEAR_AT || (!more && nnear > 0)) {
            lds_sync();
            // Whole rounds of SPLIT sources first where no pair is to be
            // decided (a compact box in a dense region); a loop whose lanes
            // end at different rounds costs 5 % there, the window 9 % more.
            // 64^3 particles in 300 halos: 1.55 ms with the general law
            // alone, 1.67 with every near pair decided in the loop, 1.45 so.
            int q0 = stream;
            unsigned long long window = 0ull;
            if (near_in) {
                const int full = nnear / SPLIT * SPLIT;
                const int4* const nl = nbuf + stream;
#pragma unroll 2
                for (int q = 0; q < full; q += SPLIT) pp_pair<false>(B, ox, oy, oz, nl[q], ngx, ngy, ngz, nph);
                q0 += full;
            }
#pragma unroll 2
            for (int q = q0; q < nnear; q += SPLIT) {
                pp_pair_cut(B, ox, oy, oz, nbuf[q], window, ngx, ngy, ngz, nph);
            }
            if (window)
                for (int q = q0; q < nnear; q += SPLIT) pp_pair_open(B, ox, oy, oz, nbuf[q], ngx, ngy, ngz, nph);
            executed += (unsigned long long)nnear * (unsigned long long)nact;
            nnear = 0;
            lds_sync();
        }
        if (!more) break;
    }
    // box units: pp_pair's sums and pp_far's offsets are in 2^-32 units
    gx = fmaf(ngx, 0x1p64f, gx * B.far_g);
    gy = fmaf(ngy, 0x1p64f, gy * B.far_g);
    gz = fmaf(ngz, 0x1p64f, gz * B.far_g);
    ph = fmaf(nph, 0x1p32f, -ph * B.far_ph);
}

// kick_pme's sums of one tile: every particle of the 27 cells by the general
// law, exact integer differences, in the cells' order.  (The far law is three times
// nearer to the FP64 sums here, 1.0e-5 of the z force's rms instead of 3.0e-5 at
// 60^3 with displacements of 0.3 cells, and takes 12.6 instead of 15.2 ms at 60^3.
// But with no cutoff a sink's sum is a small difference of large parts, whose rounding
// depends on each step of the sum: the forces moved by up to 2.6e-5, more than results may.)
template <int TS, class Sync>
__device__ __forceinline__ void pp_sum_pme(const PPArgs& a, const tpm_box_dev& B, int cx, int cy, int cz, int ox,
                                           int oy, int oz, uint32_t rx, uint32_t ry, uint32_t rz, int nact,
                                           int4* __restrict__ sbuf, Sync lds_sync, float& gx, float& gy, float& gz,
                                           float& ph, unsigned long long& executed) {
    constexpr int SPLIT = 64 / TS;
    constexpr int FLUSH_AT = 128;
    static_assert(FLUSH_AT + 64 + 2 * SPLIT <= FAR_CAP + NEAR_CAP, "room for the source read ahead");
    const int lane = (int)lane_id(), stream = lane / TS;
    const int C = B.C;
    int nbuf = 0;
    gx = gy = gz = ph = 0.f;
    auto flush = [&]() {
        // whole rounds of SPLIT sources, the next one read ahead, then the
        // streams that still have one (no padding source: the law has no cutoff)
        const int full = nbuf / SPLIT * SPLIT;
        lds_sync();
        int4 s = sbuf[stream];
#pragma unroll 2
        for (int q = 0; q < full; q += SPLIT) {
            const int4 sn = sbuf[q + SPLIT + stream];
            pp_pair<true>(B, ox, oy, oz, s, gx, gy, gz, ph);
            s = sn;
        }
        if (full + stream < nbuf) pp_pair<true>(B, ox, oy, oz, s, gx, gy, gz, ph);
        executed += (unsigned long long)nbuf * (unsigned long long)nact;
        nbuf = 0;
        lds_sync();
    };
    for (int nb = 0; nb < 27; nb++) {
        int jx = cx + nb % 3 - 1, jy = cy + (nb / 3) % 3 - 1, jz = cz + nb / 9 - 1;
        jx += jx < 0 ? C : (jx >= C ? -C : 0);
        jy += jy < 0 ? C : (jy >= C ? -C : 0);
        jz += jz < 0 ? C : (jz >= C ? -C : 0);
        const int c2 = B.cell0 + (jz * C + jy) * C + jx;
        const int sb = a.cell_begin[c2], se = a.cell_begin[c2 + 1];
        for (int j0 = sb; j0 < se; j0 += 64) {
            const int j = j0 + lane;
            if (j < se)
                sbuf[nbuf + lane] = make_int4((int)(a.x[j] - rx), (int)(a.y[j] - ry), (int)(a.z[j] - rz), j);
            nbuf += min(64, se - j0);
            if (nbuf > FLUSH_AT) flush();
        }
    }
    if (nbuf > 0) flush();
    gx *= 0x1p64f;
    gy *= 0x1p64f;
    gz *= 0x1p64f;
    ph *= 0x1p32f;
}

// The same sums with per-sink source lists (16-sink tiles, culling on).
template <class Sync>
__device__ __forceinline__ void pp_sum_lists(const PPArgs& a, const tpm_box_dev& B, int cx, int cy, int cz, int ox,
                                             int oy, int oz, uint32_t rx, uint32_t ry, uint32_t rz, bool active,
                                             int4* __restrict__ sbuf, uint8_t* __restrict__ lst,
                                             float4* __restrict__ sinkf, Sync lds_sync, float& gx, float& gy,
                                             float& gz, float& ph, unsigned long long& executed) {
    const int lane = (int)lane_id(), slot = lane % 16, stream = lane / 16;
    // Tile bounding box as floats.  float(int32) rounds by <= 64 raw units, so
    // box distances below carry <= 192 units of error, inside the 512-unit
    // margin of cull2s: the test never drops a source with r < rcut to any
    // sink.
    const float lox = (float)tile_min<16>(active ? ox : INT_MAX), hix = (float)tile_max<16>(active ? ox : INT_MIN);
    const float loy = (float)tile_min<16>(active ? oy : INT_MAX), hiy = (float)tile_max<16>(active ? oy : INT_MIN);
    const float loz = (float)tile_min<16>(active ? oz : INT_MAX), hiz = (float)tile_max<16>(active ? oz : INT_MIN);
    const int C = B.C;
    const float cull2s = B.cull2s;
    int nbuf = 0;
    gx = gy = gz = ph = 0.f;
    // Far dummy of the per-sink lists: offset -2^31 on every
    // axis, i.e. at least 1/2 - 1/C of the box from every sink of
    // the tile (a sink lies within one cell of the tile's first
    // particle), so r > rcut whenever culling is on (C >= 5).
    const int4 far = make_int4(INT_MIN, INT_MIN, INT_MIN, -1);
    // Per-sink lists: the tile's sinks as floats in LDS, read by
    // every lane alike (an inactive sink sits far from every
    // source: empty list).
    {
        if (lane < 16)
            sinkf[lane] = make_float4(active ? (float)ox : 3.0e9f, active ? (float)oy : 3.0e9f,
                                      active ? (float)oz : 3.0e9f, 0.f);
        if (lane == 0) sbuf[LFAR] = far;
    }
    // Sources in range of no sink cost nothing but the test: a
    // source joins sink k's list when its float distance to the
    // sink is inside the cull distance (float(int32) offsets are
    // off by <= 8 raw units here, far inside the 512-unit margin),
    // so no pair with r < rcut is dropped and the pair law's own
    // cutoff decides as before.
    auto flush_lists = [&]() {
        lds_sync();
        int cntv = 0;  // lane k < 16: entries of sink k's list
        for (int r0 = 0; r0 < nbuf; r0 += 64) {
            const int e = r0 + lane;
            // lanes past the staged sources test the far dummy,
            // which is in range of no sink
            const int4 sv = sbuf[e < nbuf ? e : LFAR];
            const float fx = (float)sv.x, fy = (float)sv.y, fz = (float)sv.z;
            // sink k's position is read from LDS in its own step
            // (48 positions kept live would cost occupancy); its
            // count lives in lane k of cntv
            auto sink_test = [&](auto kc) {
                constexpr int k = decltype(kc)::value;
                const float4 sk = sinkf[k];
                const float dx = fx - sk.x, dy = fy - sk.y, dz = fz - sk.z;
                const bool in = fmaf(dx, dx, fmaf(dy, dy, dz * dz)) < cull2s;
                const unsigned long long m = __ballot(in);
                const int base = __builtin_amdgcn_readlane(cntv, k);
                if (in) lst[k * LCAP + base + (int)count_below(m)] = (uint8_t)e;
                const int nb = base + __popcll(m);
                asm volatile("v_writelane_b32 %0, %1, %2" : "+v"(cntv) : "s"(nb), "i"(k));
            };
            static_for<16>(sink_test);
        }
        lds_sync();
        const int mycnt = __shfl(cntv, slot);
        const int mx = wave_max(cntv);
        int tot = cntv;
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) tot += __shfl_xor(tot, o);
        tot = __builtin_amdgcn_readfirstlane(tot);
        // stream s of sink k takes entries s, s + 4, ... of list k;
        // the index read one step ahead stays inside the lists'
        // slack (4 * ceil(LCAP / 4) + 3 < LCAP + 16)
        const uint8_t* my = lst + slot * LCAP + stream;
        const int steps = (mx + 3) >> 2;
        int pidx = stream;
        int4 sc = sbuf[pidx < mycnt ? (int)my[0] : LFAR];
#pragma unroll 2
        for (int i = 0; i < steps; i++) {
            const int pn = pidx + 4;
            const int4 sn = sbuf[pn < mycnt ? (int)my[4 * i + 4] : LFAR];
            pp_pair<false>(B, ox, oy, oz, sc, gx, gy, gz, ph);
            sc = sn;
            pidx = pn;
        }
        executed += (unsigned long long)tot;
        nbuf = 0;
        lds_sync();
    };
    for (int nb = 0; nb < 27; nb++) {
        int jx = cx + (nb % 3) - 1, jy = cy + (nb / 3) % 3 - 1, jz = cz + nb / 9 - 1;
        jx += (jx < 0) ? C : 0;
        jx -= (jx >= C) ? C : 0;
        jy += (jy < 0) ? C : 0;
        jy -= (jy >= C) ? C : 0;
        jz += (jz < 0) ? C : 0;
        jz -= (jz >= C) ? C : 0;
        const int c2 = B.cell0 + (jz * C + jy) * C + jx;
        const int sb = a.cell_begin[c2], se = a.cell_begin[c2 + 1];
        for (int j0 = sb; j0 < se; j0 += 64) {
            const int j = j0 + lane;
            bool keep = false;
            int4 sv = make_int4(0, 0, 0, j);
            if (j < se) {
                sv.x = (int)(a.x[j] - rx);
                sv.y = (int)(a.y[j] - ry);
                sv.z = (int)(a.z[j] - rz);
                const float fx = (float)sv.x, fy = (float)sv.y, fz = (float)sv.z;
                const float ex = fmaxf(fmaxf(lox - fx, fx - hix), 0.f);
                const float ey = fmaxf(fmaxf(loy - fy, fy - hiy), 0.f);
                const float ez = fmaxf(fmaxf(loz - fz, fz - hiz), 0.f);
                keep = fmaf(ex, ex, fmaf(ey, ey, ez * ez)) < cull2s;
            }
            const unsigned long long m = __ballot(keep);
            if (keep) sbuf[nbuf + (int)count_below(m)] = sv;
            nbuf += __popcll(m);
            if (nbuf > LFLUSH) flush_lists();
        }
    }
    if (nbuf > 0) flush_lists();
    // back to box units: g in 2^-64, phi in 2^-32
    gx *= 0x1p64f;
    gy *= 0x1p64f;
    gz *= 0x1p64f;
    ph *= 0x1p32f;
}

// WPG = tiles per workgroup, one wave each (1 or 4).  The waves of a
// workgroup run on one CU and take consecutive tiles of their XCD's run,
// mostly of one chain cell, so their source loads meet in that CU's L1;
// they share nothing else and never wait for each other.
// LISTS = true (16-sink tiles, culling on): each flush of staged sources is
// sorted into one list per sink of the sources within the cull distance of
// that sink (not of the tile's box), and each sink's 4 source streams walk
// its own list; a flush takes as many steps as its longest list.
template <int TS, bool BATCH, bool PERSIST, bool PME = false, int WPG = 1, bool LISTS = false>
// Occupancy: 8 waves per SIMD (64 VGPRs, no spills) for one box and for a
// batch (whose box record tile_box keeps in SGPRs); 7 with per-sink lists
// (72 VGPRs: at 64 the list build spills).
__global__ __launch_bounds__(64 * WPG, PERSIST ? 1 : (LISTS ? 7 : 8)) void pp_kick_kernel(PPArgs a) {
    static_assert(WPG == 1 || (WPG == 4 && !PERSIST), "several tiles per workgroup: one-shot launch only");
    static_assert(!LISTS || (TS == 16 && !PME), "per-sink lists: 16-sink tiles, kick_treepm's law");
    constexpr int SPLIT = 64 / TS;  // source streams per wave
    // staged sources: the far and near lists, or with LISTS the staged
    // sources, the sinks' lists and the sinks
    constexpr int NSB = FAR_CAP + NEAR_CAP > LSBUF + 16 + LCAP + 1 ? FAR_CAP + NEAR_CAP : LSBUF + 16 + LCAP + 1;
    __shared__ int4 sbufs[WPG][LISTS ? NSB : FAR_CAP + NEAR_CAP];
    const int wslot = WPG == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    int4* const sbuf = sbufs[wslot];
    // the staged list is written and read by the lanes of one wave
    auto lds_sync = [&]() {
        if constexpr (WPG == 1) {
            __syncthreads();
        } else {
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
            __builtin_amdgcn_wave_barrier();
        }
    };
    const int nt = *a.ntiles;
    const int per_xcd = (nt + 7) >> 3;
    const int xcd = (int)(blockIdx.x & 7);
    int q = xcd, qi = 0;  // persistent: current queue and queues visited
    int t;
    if constexpr (PERSIST) {
        t = INT_MAX;
    } else {
        const int k = (int)(blockIdx.x >> 3) * WPG + (WPG == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6));
        if (k >= per_xcd) return;
        t = xcd * per_xcd + k;
        if (t >= nt) return;
    }
    for (;;) {
        if constexpr (PERSIST) {
            // next tile: own queue first, then the others
            for (;;) {
                int k = 0;
                if (lane_id() == 0) k = atomicAdd(&a.queue[q], 1);
                k = __builtin_amdgcn_readfirstlane(__shfl(k, 0));
                t = q * per_xcd + k;
                if (t < min((q + 1) * per_xcd, nt)) break;
                if (++qi == 8) return;
                q = (xcd + qi) & 7;
            }
        }
        const int4 tile = a.tiles[t];
        const tpm_box_dev B = tile_box<BATCH>(a, tile.w);
        const int lane = (int)lane_id();
        const int slot = lane % TS;
        const int stream = lane / TS;
        const bool valid = tile.y + slot < tile.z;
        const int i = (int)a.order[valid ? tile.y + slot : tile.y];
        const uint32_t px = a.x[i], py = a.y[i], pz = a.z[i];
        const int r = a.rung[i];
        // the tile's first sink: the origin of its sinks' offsets
        const uint32_t rx = (uint32_t)__builtin_amdgcn_readfirstlane((int)px),
                       ry = (uint32_t)__builtin_amdgcn_readfirstlane((int)py),
                       rz = (uint32_t)__builtin_amdgcn_readfirstlane((int)pz);
        const bool active = valid && r >= B.min_rung;
        const unsigned long long amask = __ballot(active);
        if (amask == 0ull) {
            if constexpr (PERSIST)
                continue;
            else
                return;
        }
        {
            float gx = 0.f, gy = 0.f, gz = 0.f, ph = 0.f;
            unsigned long long executed = 0ull;
            {
                const int C = B.C;
                const int cid = tile.x - B.cell0;
                const int cx = cid % C, cy = (cid / C) % C, cz = cid / (C * C);
                const int nact = __popcll(amask & ((TS == 64) ? ~0ull : ((1ull << TS) - 1)));
                bool lists = false;
                if constexpr (LISTS) {
                    lists = B.cull != 0;
                    if (lists)
                        pp_sum_lists(a, B, cx, cy, cz, (int)(px - rx), (int)(py - ry), (int)(pz - rz), rx, ry, rz,
                                     active, sbuf, (uint8_t*)(sbuf + LSBUF + 16), (float4*)(sbuf + LSBUF), lds_sync,
                                     gx, gy, gz, ph, executed);
                }
                if constexpr (PME)
                    pp_sum_pme<TS>(a, B, cx, cy, cz, (int)(px - rx), (int)(py - ry), (int)(pz - rz), rx, ry, rz, nact,
                                   sbuf, lds_sync, gx, gy, gz, ph, executed);
                else if (!lists)
                    pp_sum<TS>(a, B, cx, cy, cz, px, py, pz, rx, ry, rz, active, nact, (float4*)sbuf,
                               sbuf + FAR_CAP, lds_sync, gx, gy, gz, ph, executed);
                // sum the source streams
#pragma unroll
                for (int o = TS; o < 64; o <<= 1) {
                    gx += __shfl_xor(gx, o);
                    gy += __shfl_xor(gy, o);
                    gz += __shfl_xor(gz, o);
                    ph += __shfl_xor(ph, o);
                }
            }
            {
                // Then the kick, by each active sink's stream-0 lane, with the
                // mesh force and potential made before the launch.  What only
                // the kick needs -- the output arrays and the epilogue's
                // constants -- is read from the argument block here, through
                // a pointer that the compiler cannot look through, and the
                // sink's index and rung are read again: kept over the pair
                // loop they take the SGPRs and VGPRs that it needs.
                using cbyte = const __attribute__((address_space(4))) char;
                using cargs = const __attribute__((address_space(4))) PPArgs;
                cbyte* args = (cbyte*)__builtin_amdgcn_kernarg_segment_ptr();
                asm volatile("" : "+s"(args));
                cargs* const la = (cargs*)args;
                const tpm_box_dev E = late_box<BATCH>(la, tile.w);
                unsigned long long* const lc = la->counters;
                const tpm_kick_out o{la->gx,
                                     la->gy,
                                     la->gz,
                                     la->pot,
                                     la->vx,
                                     la->vy,
                                     la->vz,
                                     la->rung,
                                     lc ? lc + TPM_COUNTER_STRIDE * (blockIdx.x % TPM_COUNTER_SLOTS) : nullptr};
                if (lane == 0 && o.counters) atomicAdd(&o.counters[0], executed);
                int nr = -1;
                if (active && stream == 0) {
                    const int i = (int)la->order[tile.y + slot];
                    const int r = la->rung[i];
                    float pgx = 0.f, pgy = 0.f, pgz = 0.f, pph = 0.f;
                    if (la->mesh) {
                        const float4 m = la->mesh[i];
                        pgx = m.x;
                        pgy = m.y;
                        pgz = m.z;
                        pph = m.w;
                    }
                    nr = kick_epilogue(E, la->flags, o, i, r, pgx, pgy, pgz, pph, gx, gy, gz, ph);
                }
                max_rung_update(o, nr);
            }
        }
        if constexpr (!PERSIST) return;
    }
}

// The kick alone (TPM_SKIP_PP): the epilogue of every active particle of the
// cells in [lo, hi) from its mesh term, one lane per particle (through
// 16-sink tiles, with a quarter of the lanes, it took 0.44 ms at 256^3).  One
// wave per cell for its first KO_RUN particles; those beyond, of crowded
// cells, KO_RUN at a time by further waves, one per KO_RUN particles of all:
// wave v looks at the cell that holds particle v KO_RUN.  (10^5 particles in
// one cell took one wave 314 us, now 10; 1024 instead of 2048 costs 256^3
// uniform ones 8 us of 115.)
#define KO_RUN 2048
template <bool BATCH>
__global__ __launch_bounds__(256) void kick_only_kernel(PPArgs a, int ncell, int nrun, int nbox, int3 lo, int3 hi) {
    const int lane = (int)lane_id();
    const int wave = __builtin_amdgcn_readfirstlane((int)((blockIdx.x * (int64_t)blockDim.x + threadIdx.x) >> 6));
    const int nwave = (int)(((int64_t)gridDim.x * blockDim.x) >> 6);
    unsigned long long* const cnt =
        a.counters ? a.counters + TPM_COUNTER_STRIDE * (blockIdx.x % TPM_COUNTER_SLOTS) : nullptr;
    const tpm_kick_out o{a.gx, a.gy, a.gz, a.pot, a.vx, a.vy, a.vz, a.rung, cnt};
    int nr = -1;
    for (int u = wave; u < ncell + nrun; u += nwave) {
        int c = u, b, e;
        if (u < ncell) {
            b = a.cell_begin[c];
            e = min(a.cell_begin[c + 1], b + KO_RUN);
        } else {
            const int i0 = (u - ncell) * KO_RUN;
            if (i0 >= a.cell_begin[ncell]) continue;
            c = tpm_upper_index(ncell, i0, [&](int k) { return (int64_t)a.cell_begin[k]; });
            b = max(i0, a.cell_begin[c] + KO_RUN);
            e = min(i0 + KO_RUN, a.cell_begin[c + 1]);
        }
        if (b >= e) continue;
        int box = 0;
        if constexpr (BATCH) box = tpm_upper_index(nbox, c, [&](int k) { return (int64_t)a.boxes[k].cell0; });
        const tpm_box_dev B = tile_box<BATCH>(a, box);
        if (!BATCH) {
            const int C = B.C, x = c % C, y = (c / C) % C, z = c / (C * C);
            if (x < lo.x || x >= hi.x || y < lo.y || y >= hi.y || z < lo.z || z >= hi.z) continue;
        }
        for (int i = b + lane; i < e; i += 64) {
            const int r = a.rung[i];
            if (r < B.min_rung) continue;
            const float4 m = a.mesh ? a.mesh[i] : make_float4(0.f, 0.f, 0.f, 0.f);
            nr = max(nr, kick_epilogue(B, a.flags, o, i, r, m.x, m.y, m.z, m.w, 0.f, 0.f, 0.f, 0.f));
        }
    }
    max_rung_update(o, nr);
}

// The mesh force and potential of every active sink of one box, as the PP
// kernel's epilogue makes them, one workgroup per chain cell: the potential
// around the cell (W^3 nodes, periodic) is read once into LDS, then each
// sink's 6 x planes go in the epilogue's SPLIT = 64 / TS parts with the
// arithmetic of mesh_interp6_part on the LDS copy, the parts summed in the
// order of the epilogue's xor shuffles -- the same bits as the epilogue.  Inside
// the PP kernel the stencil's 216 scattered loads per sink took 11 ms of a
// 204 ms launch at 512^3; here each potential value is fetched once per
// neighbouring cell.  Cell k spans raw [bounds[k], bounds[k + 1]).
// One chain cell's sinks [cb, ce); r0: the cell's first stencil node per
// axis (mesh index of its lower split plane - 2).  The W^3 nodes from r0 on
// are read into LDS first; GLOBAL: the stencil is read from phi directly (a
// cell's neighbourhood larger than the LDS cube).
template <int TS, bool GLOBAL>
__device__ __forceinline__ void mesh_force_cell(float* sphi, const uint32_t* __restrict__ x,
                                                const uint32_t* __restrict__ y, const uint32_t* __restrict__ z,
                                                const int8_t* __restrict__ rung, int min_rung, int cb, int ce,
                                                const int r0[3], const float* __restrict__ phi, int M, int W,
                                                float4* __restrict__ out) {
    constexpr int SPLIT = 64 / TS;
    const int W2 = W * W;
    if (!GLOBAL && W <= M) {
        // node l = (a W + b) W + c is r0 + (a, b, c), periodic (r0 >= -2, so
        // every coordinate lies in [-2, 2M)); a thread's next node is
        // blockDim.x further on, its (a, b, c) advanced by carries instead of
        // divisions
        const int d = (int)blockDim.x, dc = d % W, db = (d / W) % W, da = d / W2;
        int l = (int)threadIdx.x, a = l / W2, b = (l / W) % W, c = l % W;
        for (; l < W2 * W; l += d) {
            int gx = r0[0] + a, gy = r0[1] + b, gz = r0[2] + c;
            gx = gx < 0 ? gx + M : (gx >= M ? gx - M : gx);
            gy = gy < 0 ? gy + M : (gy >= M ? gy - M : gy);
            gz = gz < 0 ? gz + M : (gz >= M ? gz - M : gz);
            sphi[l] = phi[((int64_t)gx * M + gy) * M + gz];
            c += dc;
            if (c >= W) {
                c -= W;
                b++;
            }
            b += db;
            if (b >= W) {
                b -= W;
                a++;
            }
            a += da;
        }
    } else {
        // W may exceed M on tiny meshes
        for (int l = (int)threadIdx.x; l < (GLOBAL ? 0 : W2 * W); l += (int)blockDim.x) {
            const int gx = (r0[0] + l / W2 + M) % M, gy = (r0[1] + (l / W) % W + M) % M,
                      gz = (r0[2] + l % W + M) % M;
            sphi[l] = phi[((int64_t)gx * M + gy) * M + gz];
        }
    }
    __syncthreads();
    const float Mf = (float)M;
    // one lane per sink: its SPLIT parts in turn, summed as the xor shuffles
    // of a wave that splits each sink over 64 / TS lanes would sum them
    // (pairs of neighbouring parts, then pairs of pairs, ...)
    for (int i = cb + (int)threadIdx.x; i < ce; i += (int)blockDim.x) {
        if (rung[i] < min_rung) continue;
        int I0[3];
        float X[3];
        interp6_origin(x[i], y[i], z[i], M, I0, X);
        const float* base = sphi + ((I0[0] - r0[0]) * W + (I0[1] - r0[1])) * W + (I0[2] - r0[2]);
        int jx[6], jy[6], jz[6];
        if (GLOBAL) {
#pragma unroll
            for (int k = 0; k < 6; k++) {
                jx[k] = (I0[0] + k + M) % M;
                jy[k] = (I0[1] + k + M) % M;
                jz[k] = (I0[2] + k + M) % M;
            }
        }
        const auto load = [&](int aa, int bb, int cc) {
            if constexpr (GLOBAL)
                return phi[((int64_t)jx[aa] * M + jy[bb]) * M + jz[cc]];
            else
                return base[(aa * W + bb) * W + cc];
        };
        float wy[6], dwy[6], wz[6], dwz[6];
        interp6_weights(X[1], wy, dwy);
        interp6_weights(X[2], wz, dwz);
        float4 part[SPLIT];
#pragma unroll
        for (int k = 0; k < SPLIT; k++) {
            float sx = 0.f, sy = 0.f, sz = 0.f, sp = 0.f;
            interp6_planes<(6 + SPLIT - 1) / SPLIT>(X, wy, dwy, wz, dwz, k, SPLIT, load, sx, sy, sz, sp);
            part[k] = make_float4(sx, sy, sz, sp);
        }
#pragma unroll
        for (int h = 1; h < SPLIT; h <<= 1)
#pragma unroll
            for (int k = 0; k < SPLIT; k += 2 * h) {
                part[k].x += part[k + h].x;
                part[k].y += part[k + h].y;
                part[k].z += part[k + h].z;
                part[k].w += part[k + h].w;
            }
        out[i] = make_float4(-part[0].x * Mf, -part[0].y * Mf, -part[0].z * Mf, part[0].w);
    }
}

// One box: cell c = (cz C + cy) C + cx spans raw [bounds[k], bounds[k + 1]);
// only the cells in [lo, hi) per axis.
template <int TS, bool GLOBAL>
__global__ __launch_bounds__(256) void mesh_force_kernel(const uint32_t* __restrict__ x,
                                                        const uint32_t* __restrict__ y,
                                                        const uint32_t* __restrict__ z,
                                                        const int8_t* __restrict__ rung, int min_rung,
                                                        const int32_t* __restrict__ cell_begin,
                                                        const uint32_t* __restrict__ bounds, int C,
                                                        const float* __restrict__ phi, int M, int W,
                                                        int3 lo, int3 hi, float4* __restrict__ out) {
    extern __shared__ float sphi[];  // W^3, z fastest
    // Each of the 8 XCDs (workgroup index mod 8) takes one contiguous run of
    // cells in an order with z fastest, the potential's fastest axis, so
    // that the workgroups running together on one XCD read neighbouring
    // cubes through its L2 (in cell-id order, x fastest, the cubes of
    // consecutive workgroups lie a megabyte apart at 512^3 and every cube
    // came from HBM: 20.7 GB per launch).
    const int nc = C * C * C, per = (nc + 7) >> 3;
    const int rk = (int)(blockIdx.x & 7u) * per + (int)(blockIdx.x >> 3);
    if (rk >= nc) return;
    const int k3[3] = {rk / (C * C), (rk / C) % C, rk % C};
    const int c = (k3[2] * C + k3[1]) * C + k3[0];
    if (k3[0] < lo.x || k3[0] >= hi.x || k3[1] < lo.y || k3[1] >= hi.y || k3[2] < lo.z || k3[2] >= hi.z) return;
    const int cb = cell_begin[c], ce = cell_begin[c + 1];
    if (cb == ce) return;
    int r0[3];
#pragma unroll
    for (int d = 0; d < 3; d++) r0[d] = (int)(((uint64_t)bounds[k3[d]] * (uint64_t)M) >> 32) - 2;
    mesh_force_cell<TS, GLOBAL>(sphi, x, y, z, rung, min_rung, cb, ce, r0, phi, M, W, out);
}

// Batched: global cell c belongs to the last box whose cell0 <= c; its split
// planes are fixed32(k / C) and its mesh starts at mesh0.
template <int TS, bool GLOBAL>
__global__ __launch_bounds__(256) void bmesh_force_kernel(const uint32_t* __restrict__ x,
                                                         const uint32_t* __restrict__ y,
                                                         const uint32_t* __restrict__ z,
                                                         const int8_t* __restrict__ rung,
                                                         const int32_t* __restrict__ cell_begin, int nbox,
                                                         const tpm_box_dev* __restrict__ boxes,
                                                         const float* __restrict__ phi, int W, int ncell,
                                                         float4* __restrict__ out) {
    extern __shared__ float sphi[];
    // per-XCD runs of the global cell space, each box's cells with z
    // fastest, as in mesh_force_kernel
    const int per = (ncell + 7) >> 3;
    const int rk = (int)(blockIdx.x & 7u) * per + (int)(blockIdx.x >> 3);
    if (rk >= ncell) return;
    const int b = tpm_upper_index(nbox, rk, [&](int k) { return (int64_t)boxes[k].cell0; });
    const tpm_box_dev& B = boxes[b];
    const int C = B.C, M = B.M, rl = rk - B.cell0;
    int k3[3];
    if (rl < C * C * C) {
        k3[0] = rl / (C * C);
        k3[1] = (rl / C) % C;
        k3[2] = rl % C;
    } else {
        k3[0] = rl % C;
        k3[1] = (rl / C) % C;
        k3[2] = rl / (C * C);
    }
    const int c = B.cell0 + (k3[2] * C + k3[1]) * C + k3[0];
    const int cb = cell_begin[c], ce = cell_begin[c + 1];
    if (cb == ce) return;
    int r0[3];
#pragma unroll
    for (int d = 0; d < 3; d++)
        r0[d] = (int)(((uint64_t)tpm_split_plane(k3[d], B.ninv) * (uint64_t)M) >> 32) - 2;
    mesh_force_cell<TS, GLOBAL>(sphi, x, y, z, rung, B.min_rung, cb, ce, r0, phi + B.mesh0, M, W, out);
}

// W_sr = sum_c n_c * sum_{27 neighbours} n_c' (exact, 64-bit integer) over
// the global cells [0, ncell); with a box table, cell c belongs to the last
// box whose cell0 <= c.
// A single box's sinks may be restricted to the cells [lo, hi).
// tiles (may be null): the cells' particles in tiles of ts, summed.
__global__ __launch_bounds__(256) void candidate_pairs_kernel(int64_t ncell, int nbox, const tpm_box_dev* __restrict__ boxes, int C0,
                                       const int32_t* __restrict__ cell_begin, unsigned long long* __restrict__ out,
                                       int ts = 1, unsigned long long* __restrict__ tiles = nullptr,
                                       int3 lo = make_int3(0, 0, 0),
                                       int3 hi = make_int3(INT_MAX, INT_MAX, INT_MAX)) {
    unsigned long long acc = 0, nt = 0;
    for (int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; c < ncell; c += (int64_t)gridDim.x * blockDim.x) {
        int C = C0;
        int64_t base = 0;
        if (boxes) {
            const int b = tpm_upper_index(nbox, c, [&](int k) { return (int64_t)boxes[k].cell0; });
            C = boxes[b].C;
            base = boxes[b].cell0;
        }
        const int l = (int)(c - base);
        const int cx = l % C, cy = (l / C) % C, cz = l / (C * C);
        if (cx < lo.x || cx >= hi.x || cy < lo.y || cy >= hi.y || cz < lo.z || cz >= hi.z) continue;
        const int nc = cell_begin[c + 1] - cell_begin[c];
        nt += (unsigned)(nc + ts - 1) / (unsigned)ts;
        int64_t s = 0;
        for (int nb = 0; nb < 27; nb++) {
            const int jx = (cx + nb % 3 - 1 + C) % C, jy = (cy + (nb / 3) % 3 - 1 + C) % C,
                      jz = (cz + nb / 9 - 1 + C) % C;
            const int64_t c2 = base + ((int64_t)jz * C + jy) * C + jx;
            s += cell_begin[c2 + 1] - cell_begin[c2];
        }
        acc += (unsigned long long)nc * (unsigned long long)s;
    }
    // One atomic per workgroup and sum: those of all workgroups go to the same
    // words, about 12 ns each (753571 cells, one per wave and sum: 295 us; 512
    // workgroups: 62).
    __shared__ unsigned long long part[4][2];
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        acc += __shfl_xor(acc, o);
        nt += __shfl_xor(nt, o);
    }
    if (lane_id() == 0) {
        part[threadIdx.x >> 6][0] = acc;
        part[threadIdx.x >> 6][1] = nt;
    }
    __syncthreads();
    if (threadIdx.x == 0) atomicAdd(out, part[0][0] + part[1][0] + part[2][0] + part[3][0]);
    if (threadIdx.x == 0 && tiles) atomicAdd(tiles, part[0][1] + part[1][1] + part[2][1] + part[3][1]);
}
// Workgroups of candidate_pairs_kernel (256 threads).
static unsigned candidate_grid(int64_t ncell) { return std::min(grid_for(ncell, 256), 512u); }

// Drift of every live particle by v * t0 of its box (fixed32, periodic):
// raw += round(v t0 2^32) mod 2^32.
__global__ void drift_kernel(int64_t n, int nbox, const tpm_box_dev* __restrict__ boxes, uint32_t* __restrict__ x,
                             uint32_t* __restrict__ y, uint32_t* __restrict__ z, const float* __restrict__ vx,
                             const float* __restrict__ vy, const float* __restrict__ vz) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const int b = tpm_upper_index(nbox, i, [&](int k) { return boxes[k].q0; });
        const double f = boxes[b].drift * 4294967296.0;
        x[i] += (uint32_t)(uint64_t)llrint((double)vx[i] * f);
        y[i] += (uint32_t)(uint64_t)llrint((double)vy[i] * f);
        z[i] += (uint32_t)(uint64_t)llrint((double)vz[i] * f);
    }
}

template <bool BATCH>
// grid = workgroups (a multiple of 8); wpg = tiles per workgroup (1 or 4;
// the persistent and kick_pme launches take one).
static void pp_launch(int ts, bool persistent, unsigned grid, hipStream_t s, const PPArgs& a, bool pme = false,
                      int wpg = 1, bool lists = false) {
    if (lists && ts == 16 && !pme) {
        if (persistent)
            pp_kick_kernel<16, BATCH, true, false, 1, true><<<grid, 64, 0, s>>>(a);
        else if (wpg == 4)
            pp_kick_kernel<16, BATCH, false, false, 4, true><<<grid, 256, 0, s>>>(a);
        else
            pp_kick_kernel<16, BATCH, false, false, 1, true><<<grid, 64, 0, s>>>(a);
        return;
    }
    if (pme) {
        switch (ts) {
            case 8: pp_kick_kernel<8, BATCH, false, true><<<grid, 64, 0, s>>>(a); break;
            case 16: pp_kick_kernel<16, BATCH, false, true><<<grid, 64, 0, s>>>(a); break;
            case 64: pp_kick_kernel<64, BATCH, false, true><<<grid, 64, 0, s>>>(a); break;
            default: pp_kick_kernel<32, BATCH, false, true><<<grid, 64, 0, s>>>(a); break;
        }
    } else if (persistent) {
        switch (ts) {
            case 8: pp_kick_kernel<8, BATCH, true><<<grid, 64, 0, s>>>(a); break;
            case 16: pp_kick_kernel<16, BATCH, true><<<grid, 64, 0, s>>>(a); break;
            case 64: pp_kick_kernel<64, BATCH, true><<<grid, 64, 0, s>>>(a); break;
            default: pp_kick_kernel<32, BATCH, true><<<grid, 64, 0, s>>>(a); break;
        }
    } else if (wpg == 4) {
        switch (ts) {
            case 8: pp_kick_kernel<8, BATCH, false, false, 4><<<grid, 256, 0, s>>>(a); break;
            case 16: pp_kick_kernel<16, BATCH, false, false, 4><<<grid, 256, 0, s>>>(a); break;
            case 64: pp_kick_kernel<64, BATCH, false, false, 4><<<grid, 256, 0, s>>>(a); break;
            default: pp_kick_kernel<32, BATCH, false, false, 4><<<grid, 256, 0, s>>>(a); break;
        }
    } else {
        switch (ts) {
            case 8: pp_kick_kernel<8, BATCH, false><<<grid, 64, 0, s>>>(a); break;
            case 16: pp_kick_kernel<16, BATCH, false><<<grid, 64, 0, s>>>(a); break;
            case 64: pp_kick_kernel<64, BATCH, false><<<grid, 64, 0, s>>>(a); break;
            default: pp_kick_kernel<32, BATCH, false><<<grid, 64, 0, s>>>(a); break;
        }
    }
}

}  // namespace

// Waves, 4 per workgroup, up to a grid that fills the chip many times over.
static unsigned wave_grid(int64_t waves) { return (unsigned)std::min<int64_t>((waves + 3) / 4, 65536); }

void tpm_box_fill(tpm_box_dev* b, const tpm_params& p, int min_rung, int first_call, double t0, double scale) {
    b->C = p.chain_dim;
    b->M = p.mesh_dim;
    b->ninv = 1.0 / p.chain_dim;
    b->cell_w = (uint32_t)((uint64_t(1) << 32) / (uint64_t)p.chain_dim);
    b->min_rung = min_rung;
    b->first_call = first_call ? 1 : 0;
    b->do_phi = p.do_phi;
    // Constants of compute_pp_interaction (kick_treepm.cu:833-853), scaled
    // to 2^-32 units: lengths x 2^32, squares x 2^64.
    const float rcut = (float)p.rcut, rs = (float)p.rs, h = (float)p.hsoft;
    const float S = 0x1p32f;
    b->rcut2s = (rcut * rcut) * (S * S);
    // Culling keeps a margin of 512 raw units over rcut (float rounding of
    // the box distance stays below ~200); off for C < 5, where a source's
    // offset from the tile origin can wrap to the far image.
    const double cull = (double)p.rcut * 4294967296.0 + 512.0;
    b->e2s = (float)(-1.4426950408889634 / (4.0 * p.rs * p.rs) / (4294967296.0 * 4294967296.0));
    b->cull2s = (float)(cull * cull);
    b->cull = p.chain_dim >= 5 ? 1 : 0;
    b->inv2rs_s = (1.0f / rs / 2.0f) / S;
    b->tsp = 2.0f / sqrtf((float)M_PI);
    // A&S 7.1.26 p and 2/sqrt(pi), each times 1 / (2 rs) in 2^-32 units
    b->p_inv2rs_s = (float)(0.3275911 / (2.0 * p.rs) / 4294967296.0);
    b->tsp_inv2rs_s = (float)(2.0 / std::sqrt(M_PI) / (2.0 * p.rs) / 4294967296.0);
    b->inv4rs2_s = (float)(1.0 / (4.0 * p.rs * p.rs) / (4294967296.0 * 4294967296.0));
    b->k3_s = (float)(4.0 / (3.0 * std::sqrt(M_PI)) / std::pow(2.0 * p.rs * 4294967296.0, 3));
    b->h2s = (h * h) * (S * S);
    const float hinv = 1.f / h;
    b->hinv_s = hinv / S;
    b->h2inv_s = (hinv * hinv) / (S * S);
    b->h3inv_s = ((hinv * hinv * hinv) / (S * S)) / S;
    // pp_far.  far_wide bounds the half width H of a box with far sources.
    // The window: an offset s of a source, o of a sink and their difference d
    // are rounded to 2^-24 of themselves, |s| <= |d| + H, |o| <= H, so an axis
    // of a pair at rcut is off by up to 2^-23 (rcut + H), r^2 by 2 sqrt(3)
    // times that over rcut, and its own arithmetic, u's product and the
    // second-order terms add less than 8 roundings of 2^-24.
    {
        const double two32 = 4294967296.0, l2e = 1.4426950408889634;
        const float fu = (float)(l2e / (4.0 * p.rs * p.rs) / (two32 * two32));
        b->far_u = fu;
        // (below C = 5 a softened pair beyond rcut, h > rcut, has always counted)
        const double cr = (b->cull ? p.rcut : std::max(p.rcut, p.hsoft)) * two32 + 2048.0;
        b->far_cull2 = (float)(cr * cr * (1.0 + 1e-6));
        const double nr = std::max(FAR_X0 * 2.0 * p.rs, p.hsoft) * two32 + 2048.0;
        b->far_near2 = std::min((float)(nr * nr * (1.0 + 1e-6)), b->far_cull2);
        const double wide = std::min(FAR_WIDE * p.rs, 0.5) * two32;
        b->far_wide = (float)wide;
        b->far_all2 = b->far_cull2;
        b->rcut2lo = b->rcut2s * (1.f - 1e-6f);
        b->rcut2hi = b->rcut2s * (1.f + 1e-6f);
        const double rc = p.rcut * two32, uc = rc * rc * (double)fu;
        const double rel = 2.0 * std::sqrt(3.0) * std::exp2(-23.0) * (rc + wide) / rc + std::exp2(-21.0);
        b->far_ulo = (float)(uc * (1.0 - rel));
        b->far_uhi = (float)(uc * (1.0 + rel));
        b->far_wrap = (float)(0x1p31 * (1.0 - 1e-5));
        b->far_g = (float)(l2e / (8.0 * p.rs * p.rs * p.rs) / two32);
        b->far_ph = (float)(1.0 / (2.0 * p.rs));
        b->rcut2i = (uint64_t)std::ceil(rc * rc);
    }
    b->GM = (float)p.GM;
    b->phi0 = (float)(p.n_total * 4.0 * M_PI * p.rs * p.rs + (35.0 / 16.0) / p.hsoft);
    b->eta = (float)p.eta;
    b->t0 = (float)t0;
    b->scale = (float)scale;
    b->hsoft = (float)p.hsoft;
    b->drift = t0;
}

// Nodes per axis of the potential around one chain cell: the sinks of cell k
// (raw [b_k, b_k+1)) take stencil nodes from mesh index (b_k M >> 32) - 2 to
// ((b_k+1 - 1) M >> 32) + 3.  0 when the largest cube exceeds 32 KiB.
int tpm_mesh_force_width(int C, int M) {
    const double ninv = 1.0 / C;
    int w = 0;
    for (int k = 0; k < C; k++) {
        const uint64_t lo = tpm_split_plane(k, ninv);
        const uint64_t hi = (k + 1 < C ? tpm_split_plane(k + 1, ninv) : (1ull << 32)) - 1;
        const int a = (int)((lo * (uint64_t)M) >> 32) - 2, b = (int)((hi * (uint64_t)M) >> 32) + 3;
        w = std::max(w, b - a + 1);
    }
    return (int64_t)w * w * w * 4 <= 32768 ? w : 0;
}

tpm_status tpm_pp_kick(tpm_ctx* ctx, int min_rung, double scale, double t0, int first_call, unsigned flags,
                       tpm_stats* stats, const tpm_cell_box* box, int64_t ntiles_box) {
    if (!ctx->chain_valid || ctx->chain_C != ctx->C || ctx->chain_tile != ctx->tile)
        return tpm_fail(ctx, TPM_ERR_STATE, "tpm_kick: chain mesh not built (call tpm_chainmesh_create)");
    const bool use_pm = !(flags & TPM_SKIP_PM);
    if (use_pm && (!ctx->pm_valid || ctx->green_M != ctx->M))
        return tpm_fail(ctx, TPM_ERR_STATE, "tpm_kick: PM mesh not computed (call tpm_gravity_long_compute)");
    if (t0 <= 0.0) return tpm_fail(ctx, TPM_ERR_INVALID, "tpm_kick: t0 must be positive");
    if (tpm_pp_sym_eligible(ctx, min_rung, flags, box)) return tpm_pp_kick_sym(ctx, scale, t0, first_call, flags, stats);
    hipStream_t s = ctx->stream;
    if (!ctx->counters) TPM_HIP(ctx, hipMalloc(&ctx->counters, sizeof(unsigned long long) * TPM_COUNTER_WORDS));
    TPM_TRY(tpm_fill_u64(ctx, ctx->counters, TPM_COUNTER_WORDS));

    PPArgs a{};
    a.x = ctx->x;
    a.y = ctx->y;
    a.z = ctx->z;
    a.vx = ctx->vx;
    a.vy = ctx->vy;
    a.vz = ctx->vz;
    a.rung = ctx->rung;
    a.gx = ctx->gx;
    a.gy = ctx->gy;
    a.gz = ctx->gz;
    a.pot = ctx->pot;
    a.cell_begin = ctx->cell_begin;
    float4* gmesh = nullptr;
    a.counters = ctx->counters;
    a.queue = nullptr;
    a.boxes = nullptr;
    a.flags = flags;
    const int64_t ncell = (int64_t)ctx->C * ctx->C * ctx->C;
    const int64_t tiles_all = ctx->n / ctx->tile + ncell + 1;
    int64_t tiles_max = tiles_all;
    // the mesh force and potential of the active sinks, made before the
    // pair kernel (LDS cube per chain cell when it fits 32 KiB)
    ctx->mesh_force_w = tpm_mesh_force_width(ctx->C, ctx->M);
    if (use_pm && ctx->n > 0) {
        const int64_t n = ctx->n;
        if (n > ctx->mesh_force_cap) {
            if (ctx->mesh_force) TPM_HIP(ctx, hipFree(ctx->mesh_force));
            ctx->mesh_force = nullptr;
            ctx->mesh_force_cap = 0;
            TPM_HIP(ctx, hipMalloc(&ctx->mesh_force, sizeof(float4) * n));
            ctx->mesh_force_cap = n;
        }
        gmesh = static_cast<float4*>(ctx->mesh_force);
    }
    int3 blo = make_int3(0, 0, 0), bhi = make_int3(INT_MAX, INT_MAX, INT_MAX);
    if (box) {
        blo = make_int3(box->lo[0], box->lo[1], box->lo[2]);
        bhi = make_int3(box->hi[0], box->hi[1], box->hi[2]);
        if (ntiles_box > tiles_max) return tpm_fail(ctx, TPM_ERR_INVALID, "tpm_kick_box: tile count");
        tiles_max = ntiles_box;
    }
    tpm_box_fill(&a.box0, ctx->p, min_rung, first_call, t0, scale);
    a.box0.cell0 = 0;
    a.box0.mesh0 = 0;
    const bool pme = (flags & TPM_KICK_PME) != 0;
    if (pme) {
        // kick_pme: every pair of the 27 cells counts, and phi starts at 0
        a.box0.cull = 0;
        a.box0.phi0 = 0.f;
    }
    a.flags = flags & (TPM_SKIP_PP | TPM_SKIP_PM | TPM_SKIP_KICK);
    a.mesh = gmesh;

    // tiles per workgroup (kick_pme's launch: one)
    const int wpg = pme ? 1 : ctx->pp_waves;
    const int64_t per_xcd = (tiles_max + 7) / 8;
    const int64_t blocks = 8 * ((per_xcd + wpg - 1) / wpg);
    if (blocks > INT_MAX) return tpm_fail(ctx, TPM_ERR_INVALID, "tpm_kick: too many tiles");
    if (!ctx->ev[0]) {
        for (int e = 0; e < 8; e++) TPM_HIP(ctx, hipEventCreate(&ctx->ev[e]));
    }
    hipEvent_t e0 = ctx->ev[2], e1 = ctx->ev[3];
    if (ctx->prof_on) {
        e0 = tpm_prof_event(ctx);
        e1 = tpm_prof_event(ctx);
        if (!e0 || !e1) return tpm_fail(ctx, TPM_ERR_HIP, "hipEventCreate failed");
        ctx->prof_pp.emplace_back(e0, e1);
    }
    TPM_HIP(ctx, hipEventRecord(e0, s));
    if (gmesh) {
        const int W = ctx->mesh_force_w;
        const size_t lds = sizeof(float) * (size_t)W * W * W;
        const unsigned nc = (unsigned)(8 * ((ncell + 7) / 8));  // 8 XCD runs
#define TPM_MF(TSV)                                                                                               \
    if (W > 0)                                                                                                  \
        mesh_force_kernel<TSV, false><<<nc, 256, lds, s>>>(ctx->x, ctx->y, ctx->z, ctx->rung, min_rung,         \
                                                           ctx->cell_begin, ctx->bounds, ctx->C, ctx->phi,      \
                                                           ctx->M, W, blo, bhi, gmesh);                         \
    else                                                                                                        \
        mesh_force_kernel<TSV, true><<<nc, 256, 0, s>>>(ctx->x, ctx->y, ctx->z, ctx->rung, min_rung,            \
                                                        ctx->cell_begin, ctx->bounds, ctx->C, ctx->phi, ctx->M, \
                                                        0, blo, bhi, gmesh)
        switch (ctx->tile) {
            case 8: TPM_MF(8); break;
            case 16: TPM_MF(16); break;
            case 32: TPM_MF(32); break;
            default: TPM_MF(64); break;
        }
#undef TPM_MF
        TPM_HIP(ctx, hipGetLastError());
    }
    if (ctx->n > 0 && (flags & TPM_SKIP_PP)) {
        const int nrun = (int)((ctx->n + KO_RUN - 1) / KO_RUN);
        kick_only_kernel<false><<<wave_grid(ncell + nrun), 256, 0, s>>>(a, (int)ncell, nrun, 1, blo, bhi);
        TPM_HIP(ctx, hipGetLastError());
    } else if (ctx->n > 0 && blocks > 0) {
        // the tiles of the active sinks (kick_pme: of every sink, so that its
        // sums do not depend on which are active)
        if (tiles_all > ctx->tiles_cap) {
            if (ctx->tiles) TPM_HIP(ctx, hipFree(ctx->tiles));
            ctx->tiles = nullptr;
            ctx->tiles_cap = 0;
            TPM_HIP(ctx, hipMalloc(&ctx->tiles, sizeof(int4) * tiles_all));
            ctx->tiles_cap = tiles_all;
        }
        tpm_tile_args t{};
        t.x = ctx->x;
        t.y = ctx->y;
        t.z = ctx->z;
        t.rung = ctx->rung;
        t.cell_begin = ctx->cell_begin;
        t.ncell = (int32_t)ncell;
        t.C = ctx->C;
        t.min_rung = min_rung;
        t.n = t.n_all = ctx->n;
        t.cell_w = a.box0.cell_w;
        t.lo = blo;
        t.hi = bhi;
        t.ts = ctx->tile;
        t.all = pme ? 1 : 0;
        t.cnt = ctx->tile_cnt;
        t.off = ctx->tile_off;
        t.part = ctx->tile_part;
        t.tiles = ctx->tiles;
        t.order = ctx->idx;
        TPM_TRY(tpm_tiles_make(ctx->err, s, t));
        a.tiles = ctx->tiles;
        a.ntiles = ctx->tile_off + ncell;
        a.order = ctx->idx;
        pp_launch<false>(ctx->tile, false, (unsigned)blocks, s, a, pme, wpg, ctx->pp_lists != 0);
        TPM_HIP(ctx, hipGetLastError());
    }
    TPM_HIP(ctx, hipEventRecord(e1, s));
    if (stats) {
        candidate_pairs_kernel<<<candidate_grid(ncell), 256, 0, s>>>(ncell, 0, nullptr, ctx->C, ctx->cell_begin,
                                                                    ctx->counters + 2, ctx->tile,
                                                                    ctx->counters + TPM_COUNTER_TILES, blo, bhi);
        TPM_HIP(ctx, hipGetLastError());
        std::vector<unsigned long long> hw(TPM_COUNTER_WORDS);
        TPM_HIP(ctx, hipMemcpyAsync(hw.data(), ctx->counters, sizeof(unsigned long long) * TPM_COUNTER_WORDS,
                                    hipMemcpyDeviceToHost, s));
        TPM_HIP(ctx, hipStreamSynchronize(s));
        float ms = 0.f;
        TPM_HIP(ctx, hipEventElapsedTime(&ms, e0, e1));
        unsigned long long hc[4];
        tpm_reduce_counters(hw.data(), hc);
        stats->executed_pairs = (double)hc[0];
        stats->max_rung = (int)hc[1];
        stats->candidate_pairs = (double)hc[2];
        stats->ms_pp = ms;
        stats->n_tiles = (int64_t)hw[TPM_COUNTER_TILES];
    }
    return TPM_OK;
}

tpm_status tpm_candidate_pairs(tpm_ctx* ctx, unsigned long long* dst, const tpm_cell_box* box) {
    const int64_t ncell = (int64_t)ctx->C * ctx->C * ctx->C;
    int3 lo = make_int3(0, 0, 0), hi = make_int3(INT_MAX, INT_MAX, INT_MAX);
    if (box) {
        lo = make_int3(box->lo[0], box->lo[1], box->lo[2]);
        hi = make_int3(box->hi[0], box->hi[1], box->hi[2]);
    }
    candidate_pairs_kernel<<<candidate_grid(ncell), 256, 0, ctx->stream>>>(ncell, 0, nullptr, ctx->C, ctx->cell_begin,
                                                                          dst, ctx->tile,
                                                                          ctx->counters + TPM_COUNTER_TILES, lo, hi);
    TPM_HIP(ctx, hipGetLastError());
    return TPM_OK;
}

// The fused kernel over the tiles of every live box of a batch.
tpm_status tpm_batch_pp(tpm_batch* bt, const tpm_batch_layout& L, unsigned flags) {
    if (L.n_live == 0 || L.ncell == 0) return TPM_OK;
    PPArgs a{};
    a.x = bt->x;
    a.y = bt->y;
    a.z = bt->z;
    a.vx = bt->vx;
    a.vy = bt->vy;
    a.vz = bt->vz;
    a.rung = bt->rung;
    a.gx = bt->gx;
    a.gy = bt->gy;
    a.gz = bt->gz;
    a.pot = bt->pot;
    a.cell_begin = bt->cell_begin;
    a.mesh = nullptr;
    a.counters = bt->counters;
    a.queue = reinterpret_cast<int*>(bt->counters + 8);
    a.boxes = bt->d_boxes;
    a.flags = flags & (TPM_SKIP_PP | TPM_SKIP_PM | TPM_SKIP_KICK);
    if (!(flags & TPM_SKIP_PM)) {
        // the mesh force of every box's active sinks, before the pair kernel
        const size_t lds = sizeof(float) * (size_t)L.mfw * L.mfw * L.mfw;
        const unsigned nc = (unsigned)(8 * ((L.ncell + 7) / 8));  // 8 XCD runs
#define TPM_BMF(TSV)                                                                                              \
    if (L.mfw > 0)                                                                                              \
        bmesh_force_kernel<TSV, false><<<nc, 256, lds, bt->stream>>>(bt->x, bt->y, bt->z, bt->rung,             \
                                                                     bt->cell_begin, L.nbox, bt->d_boxes,       \
                                                                     bt->phi, L.mfw, (int)L.ncell,              \
                                                                     bt->mesh_force);                           \
    else                                                                                                        \
        bmesh_force_kernel<TSV, true><<<nc, 256, 0, bt->stream>>>(bt->x, bt->y, bt->z, bt->rung,                \
                                                                  bt->cell_begin, L.nbox, bt->d_boxes, bt->phi, \
                                                                  0, (int)L.ncell, bt->mesh_force)
        switch (bt->tune.tile_sinks) {
            case 8: TPM_BMF(8); break;
            case 16: TPM_BMF(16); break;
            case 32: TPM_BMF(32); break;
            default: TPM_BMF(64); break;
        }
#undef TPM_BMF
        TPM_HIP(bt, hipGetLastError());
        a.mesh = bt->mesh_force;
    }
    if (flags & TPM_SKIP_PP) {
        const int nrun = (int)((L.n_live + KO_RUN - 1) / KO_RUN);
        kick_only_kernel<true><<<wave_grid((int64_t)L.ncell + nrun), 256, 0, bt->stream>>>(
            a, L.ncell, nrun, L.nbox, make_int3(0, 0, 0), make_int3(0, 0, 0));
        TPM_HIP(bt, hipGetLastError());
        return TPM_OK;
    }
    // the tiles of every box's active sinks, their order in the sort's slot buffer
    tpm_tile_args t{};
    t.x = bt->x;
    t.y = bt->y;
    t.z = bt->z;
    t.rung = bt->rung;
    t.cell_begin = bt->cell_begin;
    t.ncell = L.ncell;
    t.nbox = L.nbox;
    t.boxes = bt->d_boxes;
    t.n_all = L.n_live;
    t.ts = bt->tune.tile_sinks;
    t.cnt = bt->tile_cnt;
    t.off = bt->tile_off;
    t.part = bt->scan_part;
    t.tiles = bt->tiles;
    t.order = bt->slot;
    TPM_TRY(tpm_tiles_make(bt->err, bt->stream, t));
    a.tiles = bt->tiles;
    a.ntiles = bt->tile_off + L.ncell;
    a.order = bt->slot;
    const bool persistent = bt->tune.sched == 1;
    int64_t grid = persistent ? bt->persist_grid : (L.tiles_max + 7) / 8 * 8;
    if (grid < 8) grid = 8;
    if (grid > INT_MAX) return tpm_fail(bt, TPM_ERR_INVALID, "tpm_batch_step: too many tiles");
    pp_launch<true>(bt->tune.tile_sinks, persistent, (unsigned)grid, bt->stream, a, false, 1, bt->tune.pp_lists != 0);
    TPM_HIP(bt, hipGetLastError());
    return TPM_OK;
}

tpm_status tpm_batch_candidates(tpm_batch* bt, const tpm_batch_layout& L) {
    if (L.ncell == 0) return TPM_OK;
    candidate_pairs_kernel<<<candidate_grid(L.ncell), 256, 0, bt->stream>>>(L.ncell, L.nbox, bt->d_boxes, 0,
                                                                           bt->cell_begin, bt->counters + 2);
    TPM_HIP(bt, hipGetLastError());
    return TPM_OK;
}

tpm_status tpm_batch_drift(tpm_batch* bt, const tpm_batch_layout& L) {
    if (L.n_live == 0) return TPM_OK;
    drift_kernel<<<grid_for(L.n_live, 256), 256, 0, bt->stream>>>(L.n_live, L.nbox, bt->d_boxes, bt->x, bt->y, bt->z,
                                                                  bt->vx, bt->vy, bt->vz);
    TPM_HIP(bt, hipGetLastError());
    return TPM_OK;
}

// Workgroups of one persistent PP launch: resident workgroups per CU x CUs,
// a multiple of the 8 XCDs.
int tpm_pp_persistent_grid(int device, int ts, bool lists) {
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, device) != hipSuccess) return 0;
    int per_cu = 0;
    hipError_t e;
    if (lists && ts == 16) {
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, pp_kick_kernel<16, true, true, false, 1, true>, 64, 0);
        if (e != hipSuccess || per_cu < 1) per_cu = 8;
        const int g = per_cu * prop.multiProcessorCount;
        return (g + 7) / 8 * 8;
    }
    switch (ts) {
        case 8: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, pp_kick_kernel<8, true, true>, 64, 0); break;
        case 16: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, pp_kick_kernel<16, true, true>, 64, 0); break;
        case 64: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, pp_kick_kernel<64, true, true>, 64, 0); break;
        default: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, pp_kick_kernel<32, true, true>, 64, 0); break;
    }
    if (e != hipSuccess || per_cu < 1) per_cu = 8;
    const int g = per_cu * prop.multiProcessorCount;
    return (g + 7) / 8 * 8;
}

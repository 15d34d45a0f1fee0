// Device side of the cell-segment decomposition: staging of a segment's
// neighbourhood union in LDS (shared by the neighbour-list build and the pair
// force kernels, which must agree slot for slot).
//
// A segment is S cells along x by R rows along y in one z-plane.  Its union
// holds 3 (R + 2) rows (dz outer, then y), each the cells x0 - 1 .. x0 + S of
// one (y, z) row; a particle's 9 candidate rows (dz, dy) are 9 of them, in
// the same (dz, dy) order.
#pragma once

#include "kernels.hpp"

namespace halmd {

constexpr unsigned SEG_CHUNKS = SEG_MAX_RECORDS / WAVE + SEG_NR;   // most 64-record chunks of a union's rows

struct seg_stage {
    seg_place q;
    unsigned nr;                            // union rows, 3 (h + 2)
    unsigned chunks;                        // 64-record chunks of the union rows
    unsigned base[SEG_NR + 1];              // LDS start of each union row; base[nr] = U
    uint4 row[SEG_NR];                      // memory ranges of each union row: begin, length, begin, length
    uint16_t chunk[SEG_CHUNKS];             // row | 256 (chunk of the row)
    unsigned own_begin[SEG_RMAX];           // memory start of the segment's particles in row j
    unsigned own_pre[SEG_RMAX + 1];         // particles of rows before j; own_pre[h] .. own_pre[SEG_RMAX] = all
};

constexpr unsigned SEG_BOUND = SEG_MAX + 3;   // bound words per union row

__device__ __forceinline__ unsigned seg_row_start(seg_params const& sp, seg_place const& q, unsigned ur) {
    unsigned const nx = sp.grid.ncell[0], ny = sp.grid.ncell[1], nz = sp.grid.ncell[2];
    unsigned const hh = q.h + 2;
    unsigned const kz = (q.z + nz + ur / hh - 1) % nz, ky = (q.y0 + ny + ur % hh - 1) % ny;
    return (kz * ny + ky) * nx;
}

// own particle t (0 .. own_pre[h] - 1) of the segment: its row j and memory index
__device__ __forceinline__ void seg_own(seg_stage const& st, unsigned t, unsigned& j, unsigned& i) {
    unsigned r = 0;
#pragma unroll
    for (unsigned k = 1; k < SEG_RMAX; ++k) r += t >= st.own_pre[k] ? 1u : 0u;   // (own_pre[k] > t from k = h on)
    j = r;
    i = st.own_begin[r] + (t - st.own_pre[r]);
}

// the largest of the DISP_SLOTS displacement words at slots exceeds bits
// (false without slots).  Each wave reads the 64 words itself, so the
// decision is uniform without a barrier.  publish (optional): lane 0 of
// workgroup 0 stores (seq << 32) | the largest word into publish[seq %
// PUBLISH_RING], host-mapped memory, by a vector store at system scope.
__device__ __forceinline__ bool displacement_aborts(uint32_t const* __restrict__ slots, uint32_t bits,
                                                    unsigned long long* publish = nullptr, uint32_t seq = 0) {
    if (!slots) return false;
    static_assert(DISP_SLOTS == WAVE, "one displacement slot per lane");
    unsigned const m = wave_max_u32(slots[(threadIdx.x % WAVE) * DISP_STRIDE]);
    if (publish && blockIdx.x == 0 && threadIdx.x == 0)
        __hip_atomic_store(publish + seq % PUBLISH_RING, (static_cast<unsigned long long>(seq) << 32) | m,
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    return m > bits;
}

// Staged record formats: the full fixed-point record (pair forces; non-cubic
// list build), or for the cubic-box list build the top 16 bits of the x and y
// coordinates in one word (x low) and of z with the species above them in the
// other.
__device__ __forceinline__ uint2 pack_rec16(uint4 const r) {
    return make_uint2((r.x >> 16) | (r.y & 0xffff0000u), (r.z >> 16) | ((r.w & 3u) << 16));
}
__device__ __forceinline__ void put_rec(uint4* s, unsigned k, uint4 const r) { s[k] = r; }
__device__ __forceinline__ void put_rec(uint2* s, unsigned k, uint4 const r) { s[k] = pack_rec16(r); }

// Called by the whole workgroup (at least 64 threads).  Fills st (and, if
// bound is given, the LDS start of each of the w + 2 cells of every union row:
// bound[ur * bstride + k], k = 0 .. w + 2; bstride >= w + 3), then, if U + 1 <= sp.lds_cap,
// copies the union into slots 0 .. U - 1 of s_rec (by put_rec, in its format) and
// a sentinel record into slot U:
// fixed-point y and z half a box from the centre of the segment's rows and
// plane, hence at least one cell width (>= rc + skin) from each of its
// particles in both (h <= ny - 2, nz >= 3).  Returns the union size U; every
// thread sees the same value.
//
// Bound: latency.  A workgroup's time is a chain of dependent memory round
// trips (about 1 us each from another XCD's writes), and below some 10^5
// particles every workgroup of the launch runs at the same time, so the chain
// is the kernel's time.  Here it is: cell offsets, records, done.  Wave 0
// locates the segment and loads the offsets of its rows in one batch (lanes
// 0 .. nr - 1 the union rows, lanes 32 .. 32 + h - 1 the own rows; no
// division, no branch), forms the prefix sums by DPP scans and lists the
// 64-record chunks of the rows; then the waves take the chunks in turn, four
// loads in flight per lane.
template <class Rec>
__device__ __forceinline__ unsigned stage_union(seg_params const& sp, unsigned seg, uint32_t const* __restrict__ off,
                                                uint4 const* __restrict__ posq, Rec* s_rec, seg_stage& st,
                                                unsigned* bound, unsigned bstride = SEG_BOUND) {
    unsigned const tid = threadIdx.x, lane = tid % WAVE;
    unsigned const nx = sp.grid.ncell[0], ny = sp.grid.ncell[1], nz = sp.grid.ncell[2];
    if (tid < WAVE) {
        seg_place const q = seg_locate(sp, seg);
        unsigned const hh = q.h + 2, nr = 3 * hh;   // <= SEG_NR = 30 < 32
        bool const own = lane >= 32 && lane < 32 + q.h, row = lane < nr;
        unsigned const dz = own ? 1u : (lane >= hh ? 1u : 0u) + (lane >= 2 * hh ? 1u : 0u);
        unsigned const dy = own ? lane - 31 : lane - dz * hh;
        unsigned const z = q.z + dz, y = q.y0 + dy;   // one more than the (periodic) coordinate
        unsigned const kz = z == 0 ? nz - 1 : (z > nz ? 0u : z - 1), ky = y == 0 ? ny - 1 : (y > ny ? 0u : y - 1);
        unsigned const first = row || own ? (kz * ny + ky) * nx : 0u;
        // cells x0 - 1 .. x0 + w (periodic) as two ranges of cells, the second
        // empty away from the box's edge in x
        bool const low = q.x0 == 0, high = q.x0 + q.w >= nx;
        unsigned const a0 = own ? q.x0 : (low ? nx - 1 : q.x0 - 1);
        unsigned const e0 = own ? q.x0 + q.w : (low || high ? nx : q.x0 + q.w + 1);
        unsigned const e1 = own ? 0u : (low ? q.w + 1 : (high ? 1u : 0u));
        unsigned const g0 = off[first + a0], h0 = off[first + e0], g1 = off[first], h1 = off[first + e1];
        unsigned const n = row || own ? (h0 - g0) + (h1 - g1) : 0u;
        unsigned const rsum = wave_inclusive_sum(row ? n : 0u);   // lanes >= nr carry the total U
        unsigned const osum = wave_inclusive_sum(own ? n : 0u);   // (lanes >= 32 + h the total)
        unsigned const c = row ? (n + WAVE - 1) / WAVE : 0u;
        unsigned const csum = wave_inclusive_sum(c);
        if (row) {
            st.base[lane] = rsum - n;
            st.row[lane] = make_uint4(g0, h0 - g0, g1, h1 - g1);
            for (unsigned k = 0; k < c && csum - c + k < SEG_CHUNKS; ++k)
                st.chunk[csum - c + k] = uint16_t(lane | k << 8);
        }
        if (lane == nr) st.base[nr] = rsum;
        if (lane >= 32 && lane < 32 + SEG_RMAX) {
            st.own_begin[lane - 32] = g0;
            st.own_pre[lane - 32 + 1] = osum;
        }
        if (lane == 63) {
            st.q = q;
            st.nr = nr;
            st.chunks = csum;
            st.own_pre[0] = 0;
        }
    }
    __syncthreads();
    seg_place const q = st.q;
    unsigned const nr = st.nr, U = st.base[nr];
    if (bound) {
        // LDS start of cell x0 - 1 + k (periodic) of union row ur, one thread each
        unsigned const nk = q.w + 3, hh = q.h + 2;
        for (unsigned e = tid; e < nr * nk; e += blockDim.x) {
            unsigned const ur = e / nk, k = e - ur * nk;
            uint4 const r = st.row[ur];
            unsigned const dz = (ur >= hh ? 1u : 0u) + (ur >= 2 * hh ? 1u : 0u);
            unsigned const z = q.z + dz, y = q.y0 + ur - dz * hh;
            unsigned const kz = z == 0 ? nz - 1 : (z > nz ? 0u : z - 1), ky = y == 0 ? ny - 1 : (y > ny ? 0u : y - 1);
            unsigned const first = (kz * ny + ky) * nx;
            unsigned const in0 = q.x0 == 0 ? 1u : min(q.w + 2, nx - q.x0 + 1);   // cells of the first range
            unsigned const cell = k <= in0 ? (q.x0 == 0 ? nx - 1 : q.x0 - 1) + k : k - in0;
            unsigned const o = off[first + cell];
            bound[ur * bstride + k] = st.base[ur] + (k <= in0 ? o - r.x : r.y + (o - r.z));
        }
    }
    if (U + 1 <= sp.lds_cap) {
        if (tid == 0) {
            // (any point about half a box away does: FP32)
            uint32_t const cy = uint32_t(float(2 * q.y0 + q.h) * (0.5f / float(ny)) * 4294967040.0f);
            uint32_t const cz = uint32_t(float(2 * q.z + 1) * (0.5f / float(nz)) * 4294967040.0f);
            put_rec(s_rec, U, make_uint4(0u, cy + 0x80000000u, cz + 0x80000000u, 0u));
        }
        unsigned const W = blockDim.x / WAVE, chunks = st.chunks;   // U <= SEG_MAX_RECORDS: every chunk is listed
        for (unsigned t = tid / WAVE; t < chunks; t += 4 * W) {   // wave-uniform
            // chunks at or past the end, and slots at or past their row's,
            // read record 0 (one cached line) and store nothing; the four
            // loads are unconditional, so that they issue back to back
            uint4 a[4];
            unsigned d[4];
#pragma unroll
            for (unsigned k = 0; k < 4; ++k) {
                bool const in = t + k * W < chunks;
                unsigned const ch = st.chunk[in ? t + k * W : 0u], r = ch & 0xffu, u = (ch >> 8) * WAVE + lane;
                uint4 const rr = st.row[r];
                bool const ok = in && u < rr.y + rr.w;
                a[k] = posq[ok ? (u < rr.y ? rr.x + u : rr.z + (u - rr.y)) : 0u];
                d[k] = ok ? st.base[r] + u : ~0u;
            }
#pragma unroll
            for (unsigned k = 0; k < 4; ++k)
                if (d[k] != ~0u) put_rec(s_rec, d[k], a[k]);
        }
    }
    __syncthreads();
    return U;
}

} // namespace halmd

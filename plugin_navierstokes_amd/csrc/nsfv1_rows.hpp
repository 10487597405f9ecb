// nsfv1_rows.hpp -- row gathers whose blocks are summed by owners.
//
// A workgroup owns consecutive nodes, a lane one incidence (node, element): it
// forms the element's row block of the node in registers.  RP rows at a time,
// the lanes put their segments (one per corner) into LDS; after one barrier a
// lane per (block, row) adds the segments of its block, in element order, from
// a list of the mesh.  The alternative, rounds in which one incidence of every
// node adds into rows in LDS, leaves most lanes idle (eight rounds for
// hexahedra, up to 24 for tetrahedra) with a barrier each: a mesh of one
// workgroup took 26 us (hexahedra) where this takes about 12.
//
// Hexahedra (OUT): the owners are sorted by their number of items, so the lanes
// of a wave loop equally long (8, 4, 2 or 1 items), and the finished segments
// pass through LDS once more to be stored in the order of the CSR values.
// 56^3 cells, LPS, the whole assembly 522 us; unsorted and stored directly 533,
// sorted and stored directly (scattered 16-byte stores) 593, rounds 580 us.
// Simplices: unsorted owners store directly; 511000 tetrahedra 265 us, sorted
// 272, through LDS 300 us.  Quadrilaterals keep the rounds (four, and unpadded
// rows): 250000 LPS 91 us against 118 us.
#pragma once

#include "nsfv1_internal.hpp"

namespace nsfv1 {

constexpr int ROWS_LANES = 256;                      // incidences of a workgroup, at most
constexpr int ROWS_NODES = 255;                      // nodes
constexpr int ROWS_BLOCKS = 8 * ROWS_LANES + ROWS_NODES;

// NC values of a row segment, in 16-byte pieces where there are four
template <int NC, typename VT>
__device__ __forceinline__ void rows_put(VT* p, const VT (&x)[NC])
{
    if constexpr (NC == 4 && sizeof(VT) == 4) {
        *reinterpret_cast<float4*>(p) = make_float4(x[0], x[1], x[2], x[3]);
    } else if constexpr (NC == 4) {
        reinterpret_cast<double2*>(p)[0] = make_double2(x[0], x[1]);
        reinterpret_cast<double2*>(p)[1] = make_double2(x[2], x[3]);
    } else {
#pragma unroll
        for (int c = 0; c < NC; ++c) p[c] = x[c];
    }
}
template <int NC, typename VT>
__device__ __forceinline__ void rows_get(const VT* p, VT (&x)[NC])
{
    if constexpr (NC == 4 && sizeof(VT) == 4) {
        const float4 t = *reinterpret_cast<const float4*>(p);
        x[0] = t.x;
        x[1] = t.y;
        x[2] = t.z;
        x[3] = t.w;
    } else if constexpr (NC == 4) {
        const double2 a = reinterpret_cast<const double2*>(p)[0], b = reinterpret_cast<const double2*>(p)[1];
        x[0] = a.x;
        x[1] = a.y;
        x[2] = b.x;
        x[3] = b.y;
    } else {
#pragma unroll
        for (int c = 0; c < NC; ++c) x[c] = p[c];
    }
}

// N corners, NC unknowns a node, RP rows a pass, workgroups of at most NB lanes
template <int N, int NC, typename VT, int RP, bool OUT, int NB = ROWS_LANES>
struct OwnedRows {
    static constexpr size_t SEG = sizeof(VT) * N * RP * NB * NC;  // segments, then defects
    static_assert(SEG >= sizeof(double) * NC * NB, "the defects take the segments' place");
    static constexpr size_t BASE = (SEG + sizeof(int) * (ROWS_NODES + 1) + sizeof(uint16_t) * N * NB + NB + 15) / 16 * 16;
    // room for the finished segments of cap blocks (the most of a workgroup)
    static constexpr size_t out_bytes(int cap)
    {
        return (sizeof(VT) * NC + sizeof(uint16_t)) * cap * RP;
    }
    // cap, or 0 (segments stored as they are finished): without OUT, and where a
    // workgroup's blocks exceed the dynamic LDS limit
    static int out_cap(int cap) { return OUT && BASE + out_bytes(cap) <= 64 * 1024 ? cap : 0; }

    VT* seg;        // [corner][row][lane][NC]
    int* nfirst;    // first incidence of each node, from the workgroup's
    uint16_t* sit;  // items: lane << 3 | corner
    uint8_t* slane; // lane of each incidence
    VT* out;        // finished segments: [row][block][NC]
    uint16_t* opos; // [row][block]: where they go, in units of NC values
    int v0, nn, i0, ni, cap;
    static constexpr int OWN = 4;
    uint2 own[OWN];  // the lane's first entries, loaded before the rows are formed
    int64_t c0;      // first CSR value and blocks of the workgroup
    int nb;

    // tables of workgroup w; the first pass's barrier covers them
    __device__ __forceinline__ OwnedRows(unsigned char* smem, const RowLists& L, const KMeshPtrs& M, int w, int cap_, bool wantJ)
    {
        cap = cap_;
        out = reinterpret_cast<VT*>(smem + BASE);
        opos = reinterpret_cast<uint16_t*>(out + cap * RP * NC);
        seg = reinterpret_cast<VT*>(smem);
        nfirst = reinterpret_cast<int*>(smem + SEG);
        sit = reinterpret_cast<uint16_t*>(nfirst + ROWS_NODES + 1);
        slane = reinterpret_cast<uint8_t*>(sit + N * NB);
        v0 = L.wg_node[w];
        nn = L.wg_node[w + 1] - v0;
        i0 = M.node_inc[v0];
        ni = M.node_inc[v0 + nn] - i0;
        const int t = threadIdx.x, nt = (int)blockDim.x;
        c0 = M.rowptr[(int64_t)v0 * NC];
        nb = (int)((M.rowptr[(int64_t)(v0 + nn) * NC] - c0) / (NC * NC));
        if (wantJ)
#pragma unroll
            for (int j = 0; j < OWN; ++j) {
                const int x = t + j * nt;
                own[j] = x < nb * RP ? L.own[c0 / (NC * NC) + x / RP] : make_uint2(0u, 0u);
            }
        for (int i = t; i <= nn; i += nt) nfirst[i] = M.node_inc[v0 + i] - i0;
        for (int i = t; i < ni; i += nt) slane[i] = L.lane_of[i0 + i];
        if (wantJ)
            for (int i = t; i < N * ni; i += nt) sit[i] = L.items[(int64_t)N * i0 + i];
    }

    __device__ __forceinline__ void put(int k, int r, const VT (&x)[NC])
    {
        rows_put<NC>(seg + ((k * RP + r) * NB + (int)threadIdx.x) * NC, x);
    }

    // rows r0 .. r0 + nr - 1 of the workgroup's blocks, after the put()s of all lanes
    __device__ __forceinline__ void sum(const RowLists& L, const KMeshPtrs& M, int r0, int nr, VT* __restrict__ J, bool vec)
    {
        __syncthreads();
#pragma unroll
        for (int j = 0; j < OWN; ++j) {
            const int x = (int)threadIdx.x + j * (int)blockDim.x;
            if (x < nb * RP) add(own[j], x % RP, r0, nr, J, vec);
        }
        for (int x = (int)threadIdx.x + OWN * (int)blockDim.x; x < nb * RP; x += (int)blockDim.x)
            add(L.own[c0 / (NC * NC) + x / RP], x % RP, r0, nr, J, vec);
        __syncthreads();
        if (!OUT || cap == 0) return;
        for (int r = 0; r < nr; ++r)
            for (int x = threadIdx.x; x < nb; x += (int)blockDim.x) {
                VT s[NC];
                rows_get<NC>(out + (r * cap + x) * NC, s);
                store(J + c0 + opos[r * cap + x] * NC, s, vec);
            }
        // the next pass puts segments beside these reads; its sums wait for a barrier
    }

    // row r of the pass of one block
    __device__ __forceinline__ void add(const uint2 o, int r, int r0, int nr, VT* __restrict__ J, bool vec)
    {
        if (r >= nr) return;
        const uint16_t* it = sit + (o.x & 0xfff);
        const int cnt = (o.x >> 12) & 0x7ff;
        VT s[NC], y[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) s[c] = VT(0);
#pragma unroll 4
        for (int i = 0; i < cnt; ++i) {
            const int z = it[i];
            rows_get<NC>(seg + (((z & 7) * RP + r) * NB + (z >> 3)) * NC, y);
#pragma unroll
            for (int c = 0; c < NC; ++c) s[c] += y[c];
        }
        const int at = (int)(o.y & 0xffff) + (r0 + r) * (int)(o.x >> 23);
        if (!OUT || cap == 0) {
            store(J + c0 + at * NC, s, vec);
        } else {
            const int b = r * cap + (int)(o.y >> 16);
            rows_put<NC>(out + b * NC, s);
            opos[b] = (uint16_t)at;
        }
    }

    static __device__ __forceinline__ void store(VT* dst, const VT (&s)[NC], bool vec)
    {
        if (vec) {
            rows_put<NC>(dst, s);
        } else {
#pragma unroll
            for (int c = 0; c < NC; ++c) dst[c] = s[c];
        }
    }

    // defects of the workgroup's nodes; every lane calls it (active: it has an incidence)
    __device__ __forceinline__ void defect(const double (&d)[NC], bool active, double* __restrict__ out)
    {
        double* ds = reinterpret_cast<double*>(seg);
        if (active)
#pragma unroll
            for (int a = 0; a < NC; ++a) ds[a * NB + threadIdx.x] = d[a];
        __syncthreads();
        for (int x = threadIdx.x; x < nn * NC; x += (int)blockDim.x) {
            const int v = x / NC, a = x % NC;
            double s = 0.0;
#pragma unroll 4
            for (int i = nfirst[v]; i < nfirst[v + 1]; ++i) s += ds[a * NB + slane[i]];
            out[(int64_t)v0 * NC + x] = s;
        }
    }
};

}  // namespace nsfv1

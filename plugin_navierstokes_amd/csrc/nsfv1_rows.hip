// nsfv1_rows.hip -- lists of the row gathers that sum their blocks by owners
// (nsfv1_rows.hpp), built on the device once per launch plan.
#include "nsfv1_rows.hpp"

namespace nsfv1 {

// One workgroup per workgroup of the plan, one thread per node: the items of
// every block in element order, then, if asked, the owners ranked by their item
// counts.
template <int N, int NC>
__global__ void __launch_bounds__(256)
row_lists(KMeshPtrs M, const int32_t* __restrict__ wg_node, const int32_t* __restrict__ perm, uint2* __restrict__ own,
          uint16_t* __restrict__ items, uint8_t* __restrict__ lane_of, bool sorted)
{
    __shared__ uint2 so[ROWS_BLOCKS];
    __shared__ uint8_t sl[ROWS_LANES];
    __shared__ int wmax[4], wsum[4];
    const int t = threadIdx.x, v0 = wg_node[blockIdx.x], v1 = wg_node[blockIdx.x + 1];
    const int i0 = M.node_inc[v0], ni = M.node_inc[v1] - i0;
    if (t < ni) sl[perm ? perm[i0 + t] - i0 : t] = (uint8_t)t;
    __syncthreads();
    if (t < ni) lane_of[i0 + t] = sl[t];
    const int64_t b0 = M.rowptr[(int64_t)v0 * NC] / (NC * NC), b1 = M.rowptr[(int64_t)v1 * NC] / (NC * NC);
    const int v = v0 + t;
    if (v < v1) {
        const int64_t r0 = M.rowptr[(int64_t)v * NC];
        const int nb = (int)((M.rowptr[(int64_t)v * NC + 1] - r0) / NC), lb = (int)(r0 / (NC * NC) - b0);
        const int j0 = M.node_inc[v], j1 = M.node_inc[v + 1];
        for (int s = 0; s < nb; ++s) so[lb + s] = make_uint2((uint32_t)nb << 23, (uint32_t)(lb * NC + s) | (uint32_t)(lb + s) << 16);
        for (int i = j0; i < j1; ++i) {
            const uint64_t pos = M.inc_pos[i];
#pragma unroll
            for (int k = 0; k < N; ++k) so[lb + (int)((pos >> (8 * k)) & 0xff)].x += 1u << 12;
        }
        uint32_t at = (uint32_t)(N * (j0 - i0));
        for (int s = 0; s < nb; ++s) {
            const uint32_t c = (so[lb + s].x >> 12) & 0x7ff;
            so[lb + s].x |= at;
            at += c;
        }
        // the low field runs through the block's items, and back by their count
        for (int i = j0; i < j1; ++i) {
            const uint64_t pos = M.inc_pos[i];
#pragma unroll
            for (int k = 0; k < N; ++k) {
                uint32_t& o = so[lb + (int)((pos >> (8 * k)) & 0xff)].x;
                items[(int64_t)N * i0 + (o & 0xfff)] = (uint16_t)(sl[i - i0] << 3 | k);
                ++o;
            }
        }
        for (int s = 0; s < nb; ++s) so[lb + s].x -= (so[lb + s].x >> 12) & 0x7ff;
    }
    __syncthreads();
    const int nb = (int)(b1 - b0);
    if (!sorted) {
        for (int x = t; x < nb; x += (int)blockDim.x) own[b0 + x] = so[x];
        return;
    }
    // One count after the other, the largest first: every thread holds consecutive
    // blocks, so a prefix sum over the threads ranks equal counts in order.  A mesh
    // has few different counts (uniform hexahedra: 8, 4, 2 and 1); comparing every
    // pair of blocks took 3.2 ms of a plan of 96^3 cells, this 0.4 (12^3: 128, 18 us).
    constexpr int PER = (ROWS_BLOCKS + ROWS_LANES - 1) / ROWS_LANES;
    const int lane = t & 63, wave = t >> 6, per = (nb + ROWS_LANES - 1) / ROWS_LANES, x0 = t * per;
    int c[PER], base = 0, last = 0x800;
#pragma unroll
    for (int i = 0; i < PER; ++i) c[i] = i < per && x0 + i < nb ? (int)(so[x0 + i].x >> 12) & 0x7ff : -1;
    for (;;) {
        int m = -1;
#pragma unroll
        for (int i = 0; i < PER; ++i) m = c[i] < last && c[i] > m ? c[i] : m;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) m = max(m, __shfl_xor(m, o, 64));
        if (lane == 0) wmax[wave] = m;
        __syncthreads();
        m = max(max(wmax[0], wmax[1]), max(wmax[2], wmax[3]));
        if (m < 0) return;
        int mine = 0;
#pragma unroll
        for (int i = 0; i < PER; ++i) mine += c[i] == m;
        int at = mine;  // inclusive sum over the wave
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int below = __shfl_up(at, o, 64);
            at += lane >= o ? below : 0;
        }
        if (lane == 63) wsum[wave] = at;
        __syncthreads();
        at += base - mine;
        for (int w = 0; w < 4; ++w) {
            at += w < wave ? wsum[w] : 0;
            base += wsum[w];
        }
#pragma unroll
        for (int i = 0; i < PER; ++i)
            if (c[i] == m) own[b0 + at++] = so[x0 + i];
        last = m;
    }
}

hipError_t launch_row_lists(int et, const KMeshPtrs& m, const int32_t* wg_node, const int32_t* perm, int nwg, uint2* own,
                            uint16_t* items, uint8_t* lane_of, hipStream_t s)
{
    if (nwg <= 0) return hipSuccess;
    switch (et) {
    case ET_TRI: row_lists<3, 3><<<nwg, 256, 0, s>>>(m, wg_node, perm, own, items, lane_of, false); break;
    case ET_TET: row_lists<4, 4><<<nwg, 256, 0, s>>>(m, wg_node, perm, own, items, lane_of, false); break;
    case ET_HEX: row_lists<8, 4><<<nwg, 256, 0, s>>>(m, wg_node, perm, own, items, lane_of, true); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace nsfv1

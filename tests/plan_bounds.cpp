// Host build of the C API without a device: memory calls work on host memory whose
// sizes are kept, the assembly launches check the launch plan instead of running it.
// Every index that the fused row kernels (assemble_rows, assemble_rows_2d) take from
// the plan and the mesh is formed as they form it and held against the arrays' sizes,
// the LDS request and the CSR pattern.
#include <hip/hip_runtime.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <set>
#include <string>

#include "../plugin_navierstokes_amd/csrc/nsfv1_internal.hpp"
#include "../plugin_navierstokes_amd/csrc/nsfv1_solver.hpp"
#include "../plugin_navierstokes_amd/csrc/nsfv1_topo.hpp"

using namespace nsfv1;

namespace {

std::map<const char*, size_t> g_mem;
std::string g_error;
int64_t g_lanes = 0;
int64_t g_rows = -1;
int g_block = 0, g_fail_at = -1, g_allocs = 0;

void bad(const std::string& what)
{
    if (g_error.empty()) g_error = what;
}

size_t room(const void* p)
{
    const auto it = g_mem.find(static_cast<const char*>(p));
    return it == g_mem.end() ? 0 : it->second;
}

// element i of an array of the API, inside its allocation
template <typename T>
T at(const T* p, int64_t i, const char* name)
{
    if (i < 0 || (size_t)(i + 1) * sizeof(T) > room(p)) {
        bad(std::string(name) + "[" + std::to_string(i) + "] of " + std::to_string(room(p) / sizeof(T)));
        return T{};
    }
    return p[i];
}

#define AT(array, i) at(M.array, i, #array)
#define NEED(cond)                 \
    do {                           \
        if (!(cond)) bad(#cond);   \
    } while (0)

template <int ET>
void check(const KMeshPtrs& M, const int4* lane_conn, int jb, int nwg, size_t lds)
{
    using T = Topo<ET>;
    constexpr int D = T::dim, N = T::nsh, NC = D + 1, NIP = T::nip;
    const int pade = NC == 4 ? 16 / jb : 0;
    const int64_t nv = (int64_t)(room(M.xyz) / (sizeof(double) * D)), nnz = (int64_t)(room(M.colidx) / sizeof(int32_t));
    NEED(lds <= 65536 && M.block >= 64 && M.block <= 256 && M.block % 64 == 0);
    g_block = M.block;
    int last = 0;
    for (int w = 0; w < nwg && g_error.empty(); ++w) {
        const int v0 = AT(wg_node, w), v1 = AT(wg_node, w + 1), rounds = AT(wg_rounds, w);
        NEED(v0 == last && v1 > v0 && v1 <= nv);
        last = v1;
        const int64_t jbase = AT(rowptr, (int64_t)v0 * NC);
        const int jlen = (int)(AT(rowptr, (int64_t)v1 * NC) - jbase), nn = v1 - v0;
        NEED(jbase >= 0 && jlen >= 0 && jbase + jlen <= nnz);
        const int64_t dbuf = ((int64_t)(jlen + nn * pade) * jb + 15) / 16 * 16;
        NEED((size_t)(dbuf + (int64_t)nn * NC * 8) <= lds);
        const int i0 = AT(node_inc, v0), i1 = AT(node_inc, v1);
        NEED(i1 >= i0 && i1 - i0 <= M.block);
        const int4 wa = AT(wg_a, 2 * w), wb = AT(wg_a, 2 * w + 1);
        NEED(wa.x == v0 && wa.y == v1 && wa.z == i0 && wa.w == i1 && wb.z == jlen && wb.w == rounds);
        NEED(((int64_t)(uint32_t)wb.x | ((int64_t)wb.y << 32)) == jbase);
        std::set<std::pair<int, int>> taken;
        std::set<int> incs;
        for (int t = i0; t < i1 && g_error.empty(); ++t) {
            ++g_lanes;
            const int inc = AT(perm, t);
            NEED(inc >= i0 && inc < i1 && incs.insert(inc).second);
            const int e = AT(inc_elem, inc), v = AT(inc_node, inc), info = AT(inc_info, inc), kv = info & 0xff, slot = info >> 8;
            NEED(v >= v0 && v < v1 && kv < N && slot >= 0 && slot < rounds && taken.insert({v, slot}).second);
            const uint64_t pw = AT(inc_pos, inc);
            const int64_t rs = AT(rowptr, (int64_t)v * NC), re = AT(rowptr, (int64_t)(v + 1) * NC);
            const int rbase = (int)(rs - jbase) + (v - v0) * pade, rlen = (int)(AT(rowptr, (int64_t)v * NC + 1) - rs);
            const int seg = rbase + (int)(re - rs);  // end of the node's rows in LDS
            NEED(seg <= jlen + nn * pade && (NC != 4 || rbase * jb % 16 == 0));
            const int4 la = AT(lane_a, t);
            NEED(la.x == e && la.y == v && (la.z & 0xff) == kv && ((la.z >> 8) & 0xff) == slot && la.z >> 16 == rlen && la.w == rbase);
            NEED(AT(lane_pos, t) == pw);
            int lc[4] = {0, 0, 0, 0};
            if (D == 2) {
                const int4 x = at(lane_conn, t, "lane_conn");
                lc[0] = x.x, lc[1] = x.y, lc[2] = x.z, lc[3] = x.w;
            }
            NEED(AT(conn, (int64_t)e * N + kv) == v);
            for (int q = 0; q < T::cip; ++q) NEED(canon_orig_ip<ET>(kv, q) >= 0 && canon_orig_ip<ET>(kv, q) < NIP);
            (void)AT(vol, (int64_t)e * N + kv);
            (void)AT(l2inv, (int64_t)e * NIP + NIP - 1);
            (void)AT(affine, e);
            for (int k = 0; k < N; ++k) {
                const int pk = canon_perm<ET>(kv, k);
                const int c = AT(conn, (int64_t)e * N + pk);
                NEED(pk >= 0 && pk < N && c >= 0 && c < nv && (D != 2 || lc[k] == c));
                const int pos = (int)((pw >> (8 * pk)) & 0xffu) * NC;
                for (int a = 0; a < NC; ++a) {
                    const int ra = rbase + a * rlen + pos;
                    NEED(pos + NC <= rlen && ra >= rbase && ra + NC <= seg);
                    for (int b = 0; b < NC; ++b)
                        NEED(AT(colidx, rs + (int64_t)a * rlen + pos + b) == c * NC + b);
                }
            }
        }
    }
    NEED(last == nv);
}

template <int ET>
void lane_nodes(const int4* lane_a, const int32_t* conn, int64_t ninc, int4* out)
{
    constexpr int N = Topo<ET>::nsh;
    for (int64_t t = 0; t < ninc; ++t) {
        int c[4] = {0, 0, 0, 0};
        for (int k = 0; k < N; ++k) c[k] = conn[(int64_t)lane_a[t].x * N + canon_perm<ET>(lane_a[t].z & 0xff, k)];
        out[t] = make_int4(c[0], c[1], c[2], c[3]);
    }
}

}  // namespace

namespace nsfv1 {

hipError_t launch_assemble(int et, int jprec, const KMeshPtrs& m, const int4* lane_conn, const KParams&, const double*,
                           const double*, void*, double*, int*, int nwg, size_t lds, hipStream_t)
{
    const int jb = jprec / 8;
    switch (et) {
    case ET_TRI: check<ET_TRI>(m, lane_conn, jb, nwg, lds); break;
    case ET_QUAD: check<ET_QUAD>(m, lane_conn, jb, nwg, lds); break;
    case ET_TET: check<ET_TET>(m, lane_conn, jb, nwg, lds); break;
    case ET_HEX: check<ET_HEX>(m, lane_conn, jb, nwg, lds); break;
    case ET_PRISM: check<ET_PRISM>(m, lane_conn, jb, nwg, lds); break;
    }
    return hipSuccess;
}
hipError_t launch_lane_nodes(int et, const int4* lane_a, const int32_t* conn, int64_t ninc, int4* out, hipStream_t)
{
    if (et == ET_TRI) lane_nodes<ET_TRI>(lane_a, conn, ninc, out);
    else lane_nodes<ET_QUAD>(lane_a, conn, ninc, out);
    return hipSuccess;
}
hipError_t launch_row_lists(int, const KMeshPtrs&, const int32_t*, const int32_t*, int, uint2*, uint16_t*, uint8_t*, hipStream_t)
{
    return hipSuccess;
}
hipError_t launch_geometry_cache(int, const double*, const int32_t*, int64_t, int, double*, double*, uint8_t*, int*, hipStream_t)
{
    return hipSuccess;
}
// Dirichlet rows as a launch would read them
hipError_t launch_dirichlet(int, const int64_t* rowptr, const int32_t*, const int64_t* rows, int64_t nrows, void*, double*,
                            const double*, const double*, hipStream_t)
{
    g_rows = nrows;
    for (int64_t i = 0; i < nrows; ++i) at(rowptr, at(rows, i, "dir_rows") + 1, "rowptr");
    return hipSuccess;
}
bool split_supported(int, const KParams&) { return false; }
bool simplex_supported(int, int) { return false; }
hipError_t noalloc_scratch_setup(int) { return hipSuccess; }
void* noalloc_scratch(int) { return nullptr; }

}  // namespace nsfv1

extern "C" {

const char* plan_error() { return g_error.c_str(); }
int64_t plan_lanes() { return g_lanes; }
int plan_block() { return g_block; }
int64_t plan_dirichlet_rows() { return g_rows; }
// the n-th allocation from now fails (n < 0: none)
void plan_fail_allocation(int n)
{
    g_fail_at = n;
    g_allocs = 0;
}

hipError_t hipMalloc(void** p, size_t n)
{
    if (g_fail_at >= 0 && g_allocs++ == g_fail_at) {
        *p = nullptr;
        return hipErrorOutOfMemory;
    }
    *p = calloc(n, 1);
    g_mem[static_cast<char*>(*p)] = n;
    return hipSuccess;
}
hipError_t hipFree(void* p)
{
    g_mem.erase(static_cast<char*>(p));
    free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind)
{
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemset(void* d, int v, size_t n)
{
    memset(d, v, n);
    return hipSuccess;
}
hipError_t hipGetDevice(int* d)
{
    *d = 0;
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "host"; }

}  // extern "C"

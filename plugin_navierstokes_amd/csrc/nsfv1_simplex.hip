// nsfv1_simplex.hip -- FP32 assembly of triangle and tetrahedron meshes in the
// common configuration (FIELDS, one upwind object of type
// no/full/skewed/LPS, no Stokes/PAC/Peclet/exact terms): one lane per element
// evaluates every SCVF once, one lane per (node, element) forms the rows'
// contributions, and lanes that own blocks add them.
//
//   simplex_records  one lane per element, in the element's own corner order:
//     the shape gradients are constant, so they, the inverse Jacobian and the
//     state gradients are formed once for all SCVFs.  Writes the corner
//     gradients, a record of 12 floats per SCVF and the FP64 defect of every
//     corner (the SCVF fluxes already added).
//   simplex_rows     a workgroup owns consecutive nodes, a lane one incidence:
//     it forms the element's row block of the node from the record and puts
//     it into LDS, two rows at a time; then one lane per (block, row) adds the
//     contributions of its block in element order, from a list, and stores
//     the finished row segment.
//
// The contributions are added by owners in one step after one barrier: in
// rounds of the incidence slot (one lane per node active, up to 24 rounds in a
// tetrahedral mesh) the gather alone took 1.0 ms of the channel's 1.55 ms.  One
// lane per block reading the records itself was slower still (1.5 ms: every
// load of a wave touches 64 different lines).
// 96 x 48 x 48 cells of six tetrahedra less four obstacles (1.28 M elements, 233000
// nodes), LPS, mass part, by a kernel trace: records 253 us (616 MB written; FP64
// ray casts at two waves per SIMD), rows 463 us (1.4 GB fetched for 616 MB of
// records, in 16-byte pieces of 128-byte lines; 229 MB written); the call 735 us
// in that run.
#include "nsfv1_geom.hpp"
#include "nsfv1_internal.hpp"
#include "nsfv1_ray.hpp"
#include "nsfv1_rows.hpp"
#include "nsfv1_topo.hpp"

namespace nsfv1 {

// Record of an element, in 16-byte chunks.  The
// chunks of eight consecutive elements are interleaved (chunk c of the eight:
// 128 contiguous bytes), so a wave writes whole cache lines and neighbouring
// elements share them when read.
template <int ET>
struct SxRec {
    static constexpr int D = Topo<ET>::dim, N = Topo<ET>::nsh, NC = D + 1, NIP = Topo<ET>::nip;
    static constexpr int GS = D == 2 ? 2 : 4;              // values per corner gradient
    static constexpr int S = (N * GS + 3) / 4 * 4;         // after the gradients, per SCVF 12 values:
    //   normal (from -> to) and flux weight | vv, vc, sp factors, -nu rho | upwind shapes
    static constexpr int VALUES = S + 12 * NIP;
    static constexpr int DEF = VALUES / 4;                 // first chunk of the corner defects
    static constexpr int CHUNKS = DEF + (N * NC + 1) / 2;
};

// four values of a record from value i (a multiple of four)
__device__ __forceinline__ void sx_put(float4* rec, int i, double a, double b, double c, double d)
{
    rec[i / 4 * 8] = make_float4((float)a, (float)b, (float)c, (float)d);
}
__device__ __forceinline__ float4 sx_get(const float4* rec, int i) { return rec[i / 4 * 8]; }

// SCVFs at a corner: the SCVF, the other end of its edge, whether the corner is
// its `from` corner, packed for lookups by a lane's corner
template <int ET>
struct SxCorner {
    static constexpr int N = Topo<ET>::nsh, CIP = Topo<ET>::cip;
    static constexpr uint64_t pack(int what)
    {
        uint64_t r = 0;
        for (int k = 0; k < N; ++k)
            for (int q = 0; q < CIP; ++q) {
                const int ip = corner_ip<ET>(k, q);
                const int f = Topo<ET>::edge[ip][0], t = Topo<ET>::edge[ip][1];
                const int v = what == 0 ? ip : (what == 1 ? (f == k ? t : f) : (f == k ? 1 : 0));
                r |= (uint64_t)v << (3 * (3 * k + q));
            }
        return r;
    }
    static constexpr uint64_t IP = pack(0), OTHER = pack(1), FROM = pack(2);
};

template <int ET>
__device__ __forceinline__ int64_t sx_first(int64_t e)
{
    return (e >> 3) * (SxRec<ET>::CHUNKS * 8) + (e & 7);
}

// upwind of SCVF IP (upwind.cpp:52-80, 133-172, 337-430, 505-575) in the
// element's own corner order
template <int ET, int IP, int TYPE>
__device__ __forceinline__ bool sx_upwind(const double (&co)[Topo<ET>::nsh][Topo<ET>::dim], const double* ipg,
                                          const double* n, const double* sv, double (&U)[Topo<ET>::nsh], double& len,
                                          uint8_t* dec, int mode)
{
    using T = Topo<ET>;
    constexpr int D = T::dim, N = T::nsh;
    constexpr int F = T::edge[IP][0], O = T::edge[IP][1];
    len = 1.0;
    if constexpr (TYPE == UPW_NO) {
#pragma unroll
        for (int k = 0; k < N; ++k) U[k] = TabH<ET>::t.phi[IP][k];
        return true;
    } else if constexpr (TYPE == UPW_FULL) {
        const bool from = dot_nc<D>(n, sv) > 0.0;
        double c[D];
#pragma unroll
        for (int i = 0; i < D; ++i) c[i] = from ? co[F][i] : co[O][i];
#pragma unroll
        for (int k = 0; k < N; ++k) U[k] = k == F ? (from ? 1.0 : 0.0) : (k == O ? (from ? 0.0 : 1.0) : 0.0);
        len = sqrt(dist2_nc<D>(ipg, c));
        return true;
    } else {
#pragma unroll
        for (int k = 0; k < N; ++k) U[k] = 0.0;
        int best = -1, side = -1;
        double gi[3] = {0, 0, 0}, li[3] = {0, 0, 0};
        if (TYPE == UPW_SKEWED && mode == 2 && dec) {
            best = *dec;
            if (best == 255) return true;
        } else {
            if (sqrt(dot_nc<D>(sv, sv)) < 1e-14) {
                if (TYPE == UPW_SKEWED && mode == 1 && dec) *dec = 255;
                return true;
            }
            // the skewed upwind takes a decision only, so the cheaper cast in
            // reference coordinates serves; the LPS shapes follow the cut point
            // and take the reference's intersection formulas
            if constexpr (TYPE == UPW_SKEWED) ray_affine<ET>(co, ipg, sv, side, gi, li);
            if (side < 0) side_loop<ET, 0>(co, ipg, sv, side, gi, li);
            if (side < 0) return false;
        }
        if constexpr (TYPE == UPW_SKEWED) {
            if (best < 0) {
                double mn = NSFV1_DBL_MAX;
#pragma unroll
                for (int s = 0; s < T::nside; ++s) {
                    if (s != side) continue;
#pragma unroll
                    for (int j = 0; j < T::side_n[s]; ++j) {
                        const double dd = dist2_nc<D>(gi, co[T::side[s][j]]);
                        if (dd < mn) {
                            mn = dd;
                            best = T::side[s][j];
                        }
                    }
                }
                if (mode == 1 && dec) *dec = (uint8_t)best;
            }
            double c[D];
#pragma unroll
            for (int i = 0; i < D; ++i) c[i] = 0.0;
#pragma unroll
            for (int k = 0; k < N; ++k) {
                U[k] = k == best ? 1.0 : 0.0;
#pragma unroll
                for (int i = 0; i < D; ++i) c[i] = k == best ? co[k][i] : c[i];
            }
            len = sqrt(dist2_nc<D>(ipg, c));
        } else {
#pragma clang fp contract(off)
#pragma unroll
            for (int k = 0; k < N; ++k) {
                bool on = false;
#pragma unroll
                for (int s = 0; s < T::nside; ++s) on |= s == side && side_has<ET>(s, k);
                double v;
                if constexpr (ET == ET_TRI) v = k == 0 ? 1.0 - li[0] - li[1] : li[k > 0 ? k - 1 : 0];
                else v = k == 0 ? 1.0 - li[0] - li[1] - li[2] : li[k > 0 ? k - 1 : 0];
                U[k] = on ? v : 0.0;
            }
            len = sqrt(dist2_nc<D>(ipg, gi));
        }
        return true;
    }
}

// Element data shared by its SCVFs.  The sums and the old state live in LDS: with
// them in registers too, the tetrahedra spill or run one wave per SIMD.
constexpr int SX_REC_BLOCK = 128;
template <int ET>
struct SxElem {
    static constexpr int D = Topo<ET>::dim, N = Topo<ET>::nsh, NC = D + 1;
    double co[N][D], ul[N][NC], c[D], g[N][D], gv[NC][D];
    double *uo, *d;  // this lane's old velocities and defect sums in LDS, value i at i * SX_REC_BLOCK
};

template <int ET, int FAST, int IP>
__device__ __forceinline__ void sx_scvf(SxElem<ET>& E, const KParams& P, double nu, const double* __restrict__ l2,
                                        uint8_t* dec, float4* __restrict__ rec, bool wantJ, bool& oku)
{
    using T = Topo<ET>;
    using R = SxRec<ET>;
    constexpr int D = T::dim, N = T::nsh, NC = D + 1;
    if constexpr (IP < T::nip) {
        double ipg[D], n[D], me[D], sv[D], pr = 0.0;
        scvf_frame<ET, IP>(E.co, E.c, ipg, n, me);
#pragma unroll
        for (int d = 0; d < D; ++d) sv[d] = 0.0;
#pragma unroll
        for (int k = 0; k < N; ++k) {
            const double ph = TabH<ET>::t.phi[IP][k];
#pragma unroll
            for (int d = 0; d < D; ++d) sv[d] += E.ul[k][d] * ph;
            pr += ph * E.ul[k][D];
        }
        double U[N], len, up[D];
        oku &= sx_upwind<ET, IP, FAST>(E.co, ipg, n, sv, U, len, dec ? dec + IP : nullptr, P.upw_mode);
#pragma unroll
        for (int d = 0; d < D; ++d) {
            double a = 0.0;
#pragma unroll
            for (int k = 0; k < N; ++k) a += U[k] * E.ul[k][d];
            up[d] = a;
        }
        // FIELDS stabilisation, diagonal case: stabilization.cpp:122-242
        const double vv = nu * l2[IP];
        const double vc = sqrt(dot_nc<D>(sv, sv)) / len;
        double diag = vv;
        if (P.has_old) diag += P.inv_dt;
        diag += vc;
        const double idg = 1.0 / diag;
        double svel[D];
#pragma unroll
        for (int d = 0; d < D; ++d) {
            double rhs = P.has_source ? P.f[d] : 0.0;
            if (P.has_old) {
                double o = 0.0;
#pragma unroll
                for (int k = 0; k < N; ++k) o += TabH<ET>::t.phi[IP][k] * E.uo[(k * D + d) * SX_REC_BLOCK];
                rhs += o * P.inv_dt;
            }
            rhs += vv * sv[d] + vc * up[d] - E.gv[D][d] * P.inv_rho;
            svel[d] = rhs * idg;
        }
        // flux, from -> to: navier_stokes_fv1.cpp:667-777
        const double prod = dot_nc<D>(sv, n) * P.rho;
        double fl[NC];
#pragma unroll
        for (int d1 = 0; d1 < D; ++d1) {
            double a = 0.0;
#pragma unroll
            for (int d2 = 0; d2 < D; ++d2) a += E.gv[d1][d2] * n[d2];
            if (!P.laplace)
#pragma unroll
                for (int d2 = 0; d2 < D; ++d2) a += E.gv[d2][d1] * n[d2];
            fl[d1] = P.s_a * (a * (-1.0 * nu * P.rho) + pr * n[d1]) + P.s_a * (up[d1] * prod);
        }
        fl[D] = P.s_a * (dot_nc<D>(svel, n) * P.rho);
#pragma unroll
        for (int a = 0; a < NC; ++a) {
            E.d[(T::edge[IP][0] * NC + a) * SX_REC_BLOCK] += fl[a];
            E.d[(T::edge[IP][1] * NC + a) * SX_REC_BLOCK] -= fl[a];
        }
        if (wantJ) {
            constexpr int C = R::S + 12 * IP;
            sx_put(rec, C, n[0], n[1], D == 3 ? n[D - 1] : 0.0, prod);
            sx_put(rec, C + 4, vv * idg, vc * idg, -P.inv_rho * idg, -1.0 * nu * P.rho);
            sx_put(rec, C + 8, U[0], U[1], U[2], N == 4 ? U[N - 1] : 0.0);
        }
        __builtin_amdgcn_sched_barrier(0);  // one SCVF's values at a time in registers
        sx_scvf<ET, FAST, IP + 1>(E, P, nu, l2, dec, rec, wantJ, oku);
    }
}

template <int ET, int FAST>
__global__ void __launch_bounds__(SX_REC_BLOCK, 2)
simplex_records(KMeshPtrs M, KParams P, const double* __restrict__ u, const double* __restrict__ uold, int64_t ne,
                float4* __restrict__ recs, int wantJ, int* __restrict__ err)
{
    using T = Topo<ET>;
    using R = SxRec<ET>;
    constexpr int D = T::dim, N = T::nsh, NC = D + 1, NIP = T::nip;
    const int64_t e = (int64_t)blockIdx.x * SX_REC_BLOCK + threadIdx.x;
    __shared__ double lds[N * (NC + D) * SX_REC_BLOCK];
    if (e >= ne) return;  // no barrier below: every lane has its own column of lds
    SxElem<ET> E;
    E.d = lds + threadIdx.x;
    E.uo = E.d + N * NC * SX_REC_BLOCK;
#pragma unroll
    for (int k = 0; k < N; ++k) {
        const int64_t v = M.conn[e * N + k];
#pragma unroll
        for (int i = 0; i < D; ++i) E.co[k][i] = M.xyz[v * D + i];
#pragma unroll
        for (int a = 0; a < NC; ++a) E.ul[k][a] = u[v * NC + a];
#pragma unroll
        for (int i = 0; i < D; ++i)
            if (P.has_old) E.uo[(k * D + i) * SX_REC_BLOCK] = uold[v * NC + i];
#pragma unroll
        for (int a = 0; a < NC; ++a) E.d[(k * NC + a) * SX_REC_BLOCK] = 0.0;
    }
    elem_centre<ET>(E.co, E.c);
    bool okg = true, oku = true;
    {
        // shape gradients: J_ij = x_(j+1),i - x_0,i, cofactor inverse, every
        // product rounded on its own, so that a gradient component that
        // vanishes in the element's own order is exactly zero
#pragma clang fp contract(off)
        double J[D][D], K[D][D];
#pragma unroll
        for (int i = 0; i < D; ++i)
#pragma unroll
            for (int j = 0; j < D; ++j) J[i][j] = E.co[j + 1][i] - E.co[0][i];
        double det;
        if constexpr (D == 2) {
            det = J[0][0] * J[1][1] - J[0][1] * J[1][0];
            K[0][0] = J[1][1];  K[0][1] = -J[0][1];
            K[1][0] = -J[1][0]; K[1][1] = J[0][0];
        } else {
            det = J[0][0] * (J[1][1] * J[2][2] - J[1][2] * J[2][1]) - J[0][1] * (J[1][0] * J[2][2] - J[1][2] * J[2][0]) +
                  J[0][2] * (J[1][0] * J[2][1] - J[1][1] * J[2][0]);
            K[0][0] = J[1][1] * J[2][2] - J[1][2] * J[2][1];
            K[0][1] = J[0][2] * J[2][1] - J[0][1] * J[2][2];
            K[0][2] = J[0][1] * J[1][2] - J[0][2] * J[1][1];
            K[1][0] = J[1][2] * J[2][0] - J[1][0] * J[2][2];
            K[1][1] = J[0][0] * J[2][2] - J[0][2] * J[2][0];
            K[1][2] = J[0][2] * J[1][0] - J[0][0] * J[1][2];
            K[2][0] = J[1][0] * J[2][1] - J[1][1] * J[2][0];
            K[2][1] = J[0][1] * J[2][0] - J[0][0] * J[2][1];
            K[2][2] = J[0][0] * J[1][1] - J[0][1] * J[1][0];
        }
        okg = det != 0.0;
#pragma unroll
        for (int i = 0; i < D; ++i) {
            double s = 0.0;
#pragma unroll
            for (int j = 0; j < D; ++j) {
                E.g[j + 1][i] = K[j][i] / det;
                s -= E.g[j + 1][i];
            }
            E.g[0][i] = s;
        }
    }
#pragma unroll
    for (int a = 0; a < NC; ++a)
#pragma unroll
        for (int i = 0; i < D; ++i) {
            double s = 0.0;
#pragma unroll
            for (int k = 0; k < N; ++k) s += E.ul[k][a] * E.g[k][i];
            E.gv[a][i] = s;
        }
    float4* rec = recs + sx_first<ET>(e);
    if (wantJ) {
        if constexpr (D == 3) {
#pragma unroll
            for (int k = 0; k < N; ++k) sx_put(rec, 4 * k, E.g[k][0], E.g[k][1], E.g[k][D - 1], 0.0);
        } else {
            sx_put(rec, 0, E.g[0][0], E.g[0][1], E.g[1][0], E.g[1][1]);
            sx_put(rec, 4, E.g[2][0], E.g[2][1], 0.0, 0.0);
        }
    }
    uint8_t* dec = (P.upw_mode != 0 && M.upw_dec) ? M.upw_dec + e * NIP : nullptr;
    sx_scvf<ET, FAST, 0>(E, P, M.nu_elem ? M.nu_elem[e] : P.nu, M.l2inv + e * NIP, dec, rec, wantJ != 0, oku);
    if (!oku) kernel_error(err, KERR_CUT_SIDE);
    if (!okg) kernel_error(err, KERR_DEGENERATE);
    double f[(N * NC + 1) / 2 * 2];
#pragma unroll
    for (int i = 0; i < (N * NC + 1) / 2 * 2; ++i) f[i] = i < N * NC ? E.d[i * SX_REC_BLOCK] : 0.0;
#pragma unroll
    for (int q = 0; q < (N * NC + 1) / 2; ++q)
        *reinterpret_cast<double2*>(rec + (R::DEF + q) * 8) = make_double2(f[2 * q], f[2 * q + 1]);
}

// rows per pass: 32 KB of segments for 256 lanes, so four workgroups fit a CU
constexpr int SX_RP = 2;

// the row gather of nsfv1_rows.hpp from the element records, lanes in the order of
// the nodes' incidences
template <int ET>
__global__ void __launch_bounds__(256)
simplex_rows(RowLists L, KMeshPtrs M, KParams P, const double* __restrict__ u, const float4* __restrict__ recs,
             float* __restrict__ J, double* __restrict__ dout)
{
    using T = Topo<ET>;
    using R = SxRec<ET>;
    using C = SxCorner<ET>;
    constexpr int D = T::dim, N = T::nsh, NC = D + 1;
    constexpr int RP = SX_RP;
    extern __shared__ __align__(16) unsigned char smem[];
    // consecutive workgroups (shared element data) go to the same XCD
    const int w = [] {
        const int nwg = (int)gridDim.x, i = (int)blockIdx.x;
        const int per = nwg >> 3, rem = nwg & 7, x = i & 7, k = i >> 3;
        return x * per + (x < rem ? x : rem) + k;
    }();
    const bool wantJ = J != nullptr, vec = ((uintptr_t)J & 15) == 0;
    OwnedRows<N, NC, float, RP, false> rows(smem, L, M, w, 0, wantJ);
    const int inc = rows.i0 + (int)threadIdx.x;
    const bool active = (int)threadIdx.x < rows.ni;
    float B[N][NC][NC];
    double dl[NC];
#pragma unroll
    for (int a = 0; a < NC; ++a) dl[a] = 0.0;
#pragma unroll
    for (int k = 0; k < N; ++k)
#pragma unroll
        for (int a = 0; a < NC; ++a)
#pragma unroll
            for (int c = 0; c < NC; ++c) B[k][a][c] = 0.f;
    if (active) {
        const int64_t e = M.inc_elem[inc];
        const int kv = M.inc_info[inc] & 0xff;
        const float4* rec = recs + sx_first<ET>(e);
#pragma unroll
        for (int q = 0; q < (NC + 1) / 2; ++q) {
            // N NC doubles in chunks of two; a corner of a triangle starts mid-chunk
            if constexpr (NC == 4) {
                const double2 f = *reinterpret_cast<const double2*>(rec + (R::DEF + 2 * kv + q) * 8);
                dl[2 * q] = f.x;
                dl[2 * q + 1] = f.y;
            } else {
                const double* f = reinterpret_cast<const double*>(rec + R::DEF * 8);
                const int x = kv * NC + 2 * q;
                dl[2 * q] = f[(x >> 1) * 16 + (x & 1)];
                if (2 * q + 1 < NC) dl[2 * q + 1 < NC ? 2 * q + 1 : 0] = f[((x + 1) >> 1) * 16 + ((x + 1) & 1)];
            }
        }
        if (wantJ) {
            float g[N][D];
            if constexpr (D == 3) {
#pragma unroll
                for (int k = 0; k < N; ++k) {
                    const float4 x = sx_get(rec, 4 * k);
                    g[k][0] = x.x;
                    g[k][1] = x.y;
                    g[k][D - 1] = x.z;
                }
            } else {
                const float4 x = sx_get(rec, 0), y = sx_get(rec, 4);
                g[0][0] = x.x;
                g[0][1] = x.y;
                g[1][0] = x.z;
                g[1][1] = x.w;
                g[N - 1][0] = y.x;
                g[N - 1][1] = y.y;
            }
            // shape values at an SCVF's ip: one for the ends of its edge, one for the rest
            constexpr float PE = (float)TabH<ET>::t.phi[0][T::edge[0][0]];
            constexpr float PO = (float)TabH<ET>::t.phi[0][3 - T::edge[0][0] - T::edge[0][1]];
            const float s_ = (float)P.s_a, rh = (float)P.rho;
            // navier_stokes_fv1.cpp:317-593 for the SCVFs at the corner
#pragma unroll
            for (int q = 0; q < T::cip; ++q) {
                const int sh = 3 * (3 * kv + q);
                const int ip = (int)(C::IP >> sh) & 7, oth = (int)(C::OTHER >> sh) & 7;
                const float sg = ((C::FROM >> sh) & 1) ? 1.f : -1.f;
                const float4* r = rec + 3 * ip * 8;
                const float4 A = sx_get(r, R::S), F = sx_get(r, R::S + 4), Ux = sx_get(r, R::S + 8);
                const float Us[4] = {Ux.x, Ux.y, Ux.z, Ux.w};
                float n[D];
                n[0] = sg * A.x;
                n[1] = sg * A.y;
                if constexpr (D == 3) n[D - 1] = sg * A.z;
                const float pw = sg * A.w, nr = F.w;
#pragma unroll
                for (int k = 0; k < N; ++k) {
                    const float ph = (k == kv || k == oth) ? PE : PO;
                    const float Sv = F.x * ph + F.y * Us[k];
                    float gn = 0.f;
#pragma unroll
                    for (int i = 0; i < D; ++i) gn += g[k][i] * n[i];
                    const float dg = nr * gn + Us[k] * pw;
                    float cpp = 0.f;
#pragma unroll
                    for (int a = 0; a < D; ++a) {
                        B[k][a][a] += s_ * dg;
                        if (!P.laplace)
#pragma unroll
                            for (int b = 0; b < D; ++b) B[k][a][b] += s_ * (nr * g[k][a] * n[b]);
                        B[k][a][D] += s_ * (ph * n[a]);
                        B[k][D][a] += s_ * (Sv * n[a] * rh);
                        cpp += g[k][a] * F.z * n[a] * rh;
                    }
                    B[k][D][D] += s_ * cpp;
                }
            }
        }
        // mass part and source: navier_stokes_fv1.cpp:781-869
        if (P.parts & 6) {
            const double vol = M.vol[e * N + kv];
            if (P.parts & 2) {
                const double m = vol * P.rho;
                const double* uv = u + (int64_t)M.inc_node[inc] * NC;
#pragma unroll
                for (int a = 0; a < D; ++a) {
#pragma unroll
                    for (int k = 0; k < N; ++k) B[k][a][a] += k == kv ? (float)(P.s_m * m) : 0.f;
                    dl[a] += P.s_m * (uv[a] * m);
                }
            }
            if ((P.parts & 4) && P.has_source)
#pragma unroll
                for (int a = 0; a < D; ++a) dl[a] += P.s_f * (P.f[a] * vol * P.rho);
        }
    }
    if (wantJ) {
#pragma unroll
        for (int r0 = 0; r0 < NC; r0 += RP) {
#pragma unroll
            for (int k = 0; k < N; ++k)
#pragma unroll
                for (int r = 0; r < RP; ++r)
                    if (r0 + r < NC) rows.put(k, r, B[k][r0 + r < NC ? r0 + r : 0]);
            rows.sum(L, M, r0, NC - r0 < RP ? NC - r0 : RP, J, vec);
        }
    }
    if (dout) rows.defect(dl, active, dout);
}

// ---------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------
// FP64 Jacobians take the fused kernel, which keeps nothing between the lanes of
// two kernels: FP64 assemblies of one handle may overlap on several streams, in
// captured graphs and through the no-allocation entry, with the same bits
bool simplex_supported(int et, int jprec) { return (et == ET_TRI || et == ET_TET) && jprec == 32; }

int64_t simplex_record_bytes(int et, int64_t ne)
{
    const int64_t chunks = et == ET_TRI ? SxRec<ET_TRI>::CHUNKS : SxRec<ET_TET>::CHUNKS;
    return (ne + 7) / 8 * 8 * chunks * 16;
}

template <int ET>
static hipError_t launch_simplex_et(const RowLists& l, const KMeshPtrs& m, const KParams& p, const double* u,
                                    const double* uold, float* J, double* d, int* err, int64_t ne, int nwg,
                                    float4* recs, hipStream_t s)
{
    const unsigned ge = (unsigned)((ne + SX_REC_BLOCK - 1) / SX_REC_BLOCK);
    const int wj = J != nullptr;
    if (ne > 0) {
        switch (p.conv_upwind) {
        case UPW_NO: simplex_records<ET, UPW_NO><<<ge, SX_REC_BLOCK, 0, s>>>(m, p, u, uold, ne, recs, wj, err); break;
        case UPW_FULL: simplex_records<ET, UPW_FULL><<<ge, SX_REC_BLOCK, 0, s>>>(m, p, u, uold, ne, recs, wj, err); break;
        case UPW_SKEWED: simplex_records<ET, UPW_SKEWED><<<ge, SX_REC_BLOCK, 0, s>>>(m, p, u, uold, ne, recs, wj, err); break;
        case UPW_LPS: simplex_records<ET, UPW_LPS><<<ge, SX_REC_BLOCK, 0, s>>>(m, p, u, uold, ne, recs, wj, err); break;
        default: return hipErrorInvalidValue;
        }
    }
    using Rows = OwnedRows<Topo<ET>::nsh, Topo<ET>::dim + 1, float, SX_RP, false>;
    static_assert(Rows::BASE <= 64 * 1024, "dynamic LDS limit");
    if (nwg > 0) simplex_rows<ET><<<nwg, 256, Rows::BASE, s>>>(l, m, p, u, recs, J, d);
    return hipGetLastError();
}

hipError_t launch_assemble_simplex(int et, const RowLists& l, const KMeshPtrs& m, const KParams& p, const double* u,
                                   const double* uold, float* J, double* d, int* err, int64_t ne, int nwg, void* recs,
                                   hipStream_t s)
{
    float4* r = static_cast<float4*>(recs);
    if (et == ET_TRI) return launch_simplex_et<ET_TRI>(l, m, p, u, uold, J, d, err, ne, nwg, r, s);
    if (et == ET_TET) return launch_simplex_et<ET_TET>(l, m, p, u, uold, J, d, err, ne, nwg, r, s);
    return hipErrorInvalidValue;
}

}  // namespace nsfv1

// Fused element assembly kernels (p121 loop A, p123 element loop).
//
// One 64-lane wavefront builds one element: SAMPLE's 2x2x2 Gauss points,
// SHAPE_DER at each point, the jacobian, its determinant and inverse, global
// derivatives, then the element matrix, written once to HBM: as the FP64
// packed triangle (pf_internal.h; column pairs where it does not hold), or --
// for FP32 storage -- straight into the packed symmetric hi/lo layout (hi =
// fl32(K), lo = fl32(K - hi) of the upper triangle) together with the
// element's FP64 diagonal, so an FP32-stored problem never holds the FP64
// matrices.
// Nothing but the element coordinates is read and nothing but the matrix is
// written.
//
// Reference: src/programs/5th_ed/p121/p121.f90:54-64 (elastic),
// src/programs/5th_ed/p123/p123.f90:70-84 (Laplace); element routines in
// src/modules/shared/new_library.f90 (SAMPLE :1406-1433, SHAPE_DER hex8
// :769-794, hex20 :865-896, BEEMAT :976-993, DEEMAT :1671-1686) and
// src/modules/mpi/maths.f90 (INVERT :525-547, DETERMINANT :615-619).
//
// Every quantity is formed with the reference's operation order (sums in
// ascending index order, each product and sum rounded, no fused
// multiply-add), skipping only products with the structural zeros of B and
// dee, which add exact zeros.  The element matrices therefore equal the ones
// a sequential evaluation of p121's MATMUL(MATMUL(TRANSPOSE(bee),dee),bee)
// *det*weights(i) gives, bit for bit.
#include "pf_internal.h"
#include "pf_device.h"
#include "pf_element.h"

namespace {

constexpr int WAVES = 4;   // elements per block

// SAMPLE hexahedron nip=8 (new_library.f90:1406-1433): the signs of
// (xi,eta,zeta) at point g, in the reference's order, and 1/sqrt(3).
constexpr int gauss_sign[8][3] = {{1, 1, 1}, {1, 1, -1}, {1, -1, 1}, {1, -1, -1},
                                  {-1, 1, 1}, {-1, -1, 1}, {-1, 1, -1}, {-1, -1, -1}};
constexpr double gauss_r3 = 0.57735026918962584;   // the double 1.0 / sqrt(3.0)

// SHAPE_DER at every Gauss point: the same for every element, so evaluated
// once, by the compiler, with the operations of shape_der3 in their order.
template <int NOD> struct DerTable {
    double v[8][3][NOD];
    constexpr DerTable() : v()
    {
        for (int g = 0; g < 8; ++g)
            for (int l = 0; l < NOD; ++l) {
                double d[3] = {0.0, 0.0, 0.0};
                shape_der3<NOD>(gauss_sign[g][0] * gauss_r3, gauss_sign[g][1] * gauss_r3, gauss_sign[g][2] * gauss_r3, l,
                                d);
                for (int a = 0; a < 3; ++a) v[g][a][l] = d[a];
            }
    }
};
__device__ constexpr DerTable<8> der_table8{};
__device__ constexpr DerTable<20> der_table20{};
template <int NOD> __device__ __forceinline__ const double *der_at(int g, int a)
{
    if constexpr (NOD == 8) return der_table8.v[g][a];
    else return der_table20.v[g][a];
}

// Per-wave LDS scratch for one element.
template <int NOD>
struct ElemLds {
    double coord[NOD * 3];      // (nod,3) column-major, as g_coord_pp(:,:,iel)
    double jac[8][9];           // jacobian (3x3 column-major)
    double inv[8][9];           // its inverse
    double dw[8];               // det * weight
    double deriv[8][3][NOD];    // global derivatives
};

// Stages shared by the element types: jacobian, DETERMINANT/INVERT, global
// derivatives.  All waves of the block call it (block-uniform barriers);
// `valid` masks elements past the last.
template <int NOD>
__device__ __forceinline__ void element_geometry(ElemLds<NOD> &L, const double *__restrict__ gc, int lane, bool valid)
{
    if (valid)
        for (int k = lane; k < NOD * 3; k += 64) L.coord[k] = gc[k];
    __syncthreads();
    // jac = MATMUL(der, coord): 72 entries (8 points x 3 x 3).
    for (int k = lane; k < 72; k += 64) {
        const int g = k / 9, ab = k % 9, a = ab % 3, b = ab / 3;
        const double *der = der_at<NOD>(g, a);
        double s = 0.0;
#pragma unroll
        for (int l = 0; l < NOD; ++l) s += der[l] * L.coord[l + NOD * b];
        L.jac[g][a + 3 * b] = s;
    }
    __syncthreads();
    // DETERMINANT (maths.f90:615-619) and INVERT (maths.f90:525-547), an entry
    // per lane: entry (r,c) of the inverse is P - Q with P = M(c+1,r+1)
    // M(c+2,r+2) and Q = M(c+2,r+1) M(c+1,r+2), indices cyclic -- INVERT's nine
    // statements, whose -A + B and B - A round alike -- over the determinant.
    for (int k = lane; k < 72; k += 64) {
        const int g = k / 9, rc = k % 9, r = rc % 3, c = rc / 3;
        const double *m = L.jac[g];
#define M(a, b) m[((a)-1) + 3 * ((b)-1)]
        double det = M(1, 1) * (M(2, 2) * M(3, 3) - M(3, 2) * M(2, 3));
        det = det - M(1, 2) * (M(2, 1) * M(3, 3) - M(3, 1) * M(2, 3));
        det = det + M(1, 3) * (M(2, 1) * M(3, 2) - M(3, 1) * M(2, 2));
#undef M
        const int r1 = r == 2 ? 0 : r + 1, r2 = r == 0 ? 2 : r - 1, c1 = c == 2 ? 0 : c + 1, c2 = c == 0 ? 2 : c - 1;
        const double P = m[c1 + 3 * r1] * m[c2 + 3 * r2], Q = m[c2 + 3 * r1] * m[c1 + 3 * r2];
        L.inv[g][r + 3 * c] = (P - Q) / det;
        if (rc == 0) L.dw[g] = det;   // SAMPLE weights are 1 for nip = 8
    }
    __syncthreads();
    // deriv = MATMUL(jac^-1, der)
    for (int k = lane; k < 8 * NOD; k += 64) {
        const int g = k / NOD, l = k % NOD;
        const double *ji = L.inv[g];
        const double d0 = der_at<NOD>(g, 0)[l], d1 = der_at<NOD>(g, 1)[l], d2 = der_at<NOD>(g, 2)[l];
        for (int a = 0; a < 3; ++a) L.deriv[g][a][l] = ji[a] * d0 + ji[a + 3] * d1 + ji[a + 6] * d2;
    }
    __syncthreads();
}

// Elastic element.  Lane i is row i of K_e (node a = i/3, component ci).
// The entry (i,j) at a Gauss point is sum_k btd(i,k) B(k,j) with
// btd(i,k) = sum_l B(l,i) dee(l,k), evaluated in the reference's order
// (l then k ascending, every product rounded, no fused multiply-add); the
// zero entries of B and dee contribute exact zeros, so only the non-zero
// products are formed:
//   x dof: B(1,i)=dx B(4,i)=dy B(6,i)=dz   y dof: B(2,i)=dy B(4,i)=dx B(5,i)=dz
//   z dof: B(3,i)=dz B(5,i)=dy B(6,i)=dx   (BEEMAT ih=6)
// and km(i,j) += (s*det)*w with SAMPLE's w = 1.
// FP32 storage: entry (i, j), j >= i, of element e (the upper triangle the
// packed layout keeps) as hi and lo; the diagonal also in FP64 into dg(i,e)
// for the assembled Jacobi diagonal.
template <int NT>
__device__ __forceinline__ void store_packed(long e, int i, int j, double k, float *__restrict__ hi,
                                             float *__restrict__ lo, double *__restrict__ dg)
{
    if (j < i) return;
    const long t = pf_idx_sym_ij(e, NT, i, j);
    const float h = (float)k;
    hi[t] = h;
    lo[t] = (float)(k - (double)h);
    if (j == i) dg[e * NT + i] = k;
}

// Zero padding at the end of element e's packed block.
template <int NT>
__device__ __forceinline__ void zero_padding(long e, int lane, float *__restrict__ hi, float *__restrict__ lo)
{
    constexpr int used = NT * (NT + 1) / 2, pad = (int)pf_sym_per(NT) - used;
    if (lane < pad) {
        hi[e * pf_sym_per(NT) + used + lane] = 0.0f;
        lo[e * pf_sym_per(NT) + used + lane] = 0.0f;
    }
}

// Difference K(i,j) - K(j,i) as an FP16 multiple of the element's unit (inv =
// 1/unit, a power of two: both scalings are exact), and whether it brings the
// entry back exactly as the product will form it, the sign of a zero included:
// no difference is the zero of the lower entry's sign, which leaves every upper
// entry but a zero of the other sign as it is.
__device__ __forceinline__ _Float16 tri_code(double low, double up, double inv, double unit, bool &fail)
{
    const double d = __dsub_rn(low, up);
    const _Float16 h = (_Float16)(float)(d == 0.0 ? copysign(d, low) : d * inv);
    const double back = __fma_rn((double)h, unit, up);
    fail |= !(back == low) || signbit(back) != signbit(low);
    return h;
}

// The unit (its high word; inv its reciprocal) that puts an element's largest
// difference dm at [2^14, 2^15) units; false where there is none.
__device__ __forceinline__ bool tri_unit(double dm, unsigned &uh, double &unit, double &inv)
{
    const int ex = (int)((__double_as_longlong(dm) >> 52) & 0x7FF);   // dm >= 0
    const bool ok = dm == 0.0 || (ex > 14 && ex < 2046 - 14);
    uh = dm == 0.0 || !ok ? 1023u << 20 : (unsigned)(ex - 14) << 20;
    unit = __hiloint2double((int)uh, 0);
    inv = __hiloint2double((int)((2046u << 20) - uh), 0);
    return ok;
}

// Where the elastic assembly writes.
enum { AS_PAIRS = 0, AS_PACK32 = 1, AS_TRI = 2 };
struct as_out {
    double *K;                   // AS_PAIRS: column pairs; AS_TRI: the triangle
    unsigned *diff, *unit;       // AS_TRI
    int *bad;                    // AS_TRI: set where an entry does not come back exactly
    float *hi, *lo;              // AS_PACK32
    double *dg;                  // AS_PACK32, AS_TRI: element diagonals
};

// One wavefront per workgroup and element.  The row's NT entries are
// accumulated in registers, Gauss point by Gauss point: a point costs its 3 NOD
// global derivatives, read from LDS as broadcasts, once for all columns (a
// column-by-column evaluation read every derivative for every entry and kept
// B^T D of all 8 points in registers instead).  Bound by the FP64 products
// and sums, which the reference's rounding keeps apart: 21 per node and point,
// 5.5 ms for 1M hex20 elements.  The LDS of the geometry is reused to hand the
// upper triangle from the lanes that hold it to those that write it.
template <int NOD, int MODE>
__global__ __launch_bounds__(64, NOD == 20 ? 2 : 4) void k_assemble_elastic(
    const double *__restrict__ g_coord, const double *__restrict__ e_elem, double v2, double vv,
    double den, double e0, as_out O)
{
    constexpr int NT = 3 * NOD, H = NT / 2, LOW = H * (H - 1), PAIRS = H * (H + 1);
    constexpr size_t XCH = sizeof(double2) * (MODE == AS_TRI ? LOW : MODE == AS_PACK32 ? PAIRS : 1);
    constexpr size_t GEO = sizeof(ElemLds<NOD>);
    __shared__ __attribute__((aligned(16))) unsigned char raw[GEO > XCH ? GEO : XCH];
    ElemLds<NOD> &L = *reinterpret_cast<ElemLds<NOD> *>(raw);
    const int lane = threadIdx.x;
    const long e = blockIdx.x;
    element_geometry<NOD>(L, g_coord + e * (NOD * 3), lane, true);
    // DEEMAT: dee = dee0 * (e / (2(1+v)vv)) with dee0 = 1 on the normal
    // diagonal, v2 off it, vv on the shear diagonal.
    const double f = (e_elem ? e_elem[e] : e0) / den;
    const double D11 = 1.0 * f, D12 = v2 * f, D44 = vv * f;
    const int i = lane < NT ? lane : NT - 1;
    const bool on = lane < NT;
    const int a = i / 3, ci = i - 3 * a;
    double k[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) k[j] = 0.0;
#pragma unroll 1
    for (int g = 0; g < 8; ++g) {
        const double ax = L.deriv[g][0][a], ay = L.deriv[g][1][a], az = L.deriv[g][2][a];
        const double det = L.dw[g];
        // row i of B^T D at this point
        const double an = ci == 0 ? ax : ci == 1 ? ay : az;
        const double t0 = an * (ci == 0 ? D11 : D12), t1 = an * (ci == 1 ? D11 : D12), t2 = an * (ci == 2 ? D11 : D12);
        const double t3 = ci == 0 ? ay * D44 : ci == 1 ? ax * D44 : 0.0;
        const double t4 = ci == 0 ? 0.0 : ci == 1 ? az * D44 : ay * D44;
        const double t5 = ci == 0 ? az * D44 : ci == 1 ? 0.0 : ax * D44;
#pragma unroll
        for (int b = 0; b < NOD; ++b) {
            const double dx = L.deriv[g][0][b], dy = L.deriv[g][1][b], dz = L.deriv[g][2][b];
            const double sx = (t0 * dx + t3 * dy) + t5 * dz;   // column x dof of node b
            const double sy = (t1 * dy + t3 * dx) + t4 * dz;   // column y dof
            const double sz = (t2 * dz + t4 * dy) + t5 * dx;   // column z dof
            k[3 * b] = k[3 * b] + sx * det;
            k[3 * b + 1] = k[3 * b + 1] + sy * det;
            k[3 * b + 2] = k[3 * b + 2] + sz * det;
        }
    }
    __syncthreads();   // the derivatives' LDS is free
    if constexpr (MODE == AS_PAIRS) {
        double2 *Kp = reinterpret_cast<double2 *>(O.K + e * (long)(NT * NT)) + i;
        if (on)
#pragma unroll
            for (int s = 0; s < H; ++s) Kp[s * NT] = make_double2(k[2 * s], k[2 * s + 1]);
    } else if constexpr (MODE == AS_PACK32) {
        // the upper triangle through LDS (as column pairs), so that every lane
        // writes its row's packed entries K(i, i+d mod NT) as whole quads
        double2 *X = reinterpret_cast<double2 *>(raw);
#pragma unroll
        for (int s = 0; s < H; ++s)
            if (on && i <= 2 * s + 1) X[pf_tri_pair(s, i)] = make_double2(k[2 * s], k[2 * s + 1]);
        __syncthreads();
        const double *x = reinterpret_cast<const double *>(raw);
        auto entry = [&](int d) {   // K(i, i + d mod NT) from the upper triangle
            int j = i + d;
            if (j >= NT) j -= NT;
            const int r = i < j ? i : j, q = i < j ? j : i;
            return x[2 * pf_tri_pair(q >> 1, r) + (q & 1)];
        };
        constexpr int Q = pf_sym_quads(NT), RM = pf_sym_rem(NT);
        float *hi = O.hi + e * pf_sym_per(NT), *lo = O.lo + e * pf_sym_per(NT);
        if (on) {
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                float4 h, l;
                float *hp = &h.x, *lp = &l.x;
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const double v = entry(4 * q + c);
                    hp[c] = (float)v;
                    lp[c] = (float)(v - (double)hp[c]);
                }
                reinterpret_cast<float4 *>(hi)[q * NT + i] = h;
                reinterpret_cast<float4 *>(lo)[q * NT + i] = l;
            }
#pragma unroll
            for (int c = 0; c < RM; ++c) {
                const double v = entry(4 * Q + c);
                const float h = (float)v;
                hi[4 * Q * NT + RM * i + c] = h;
                lo[4 * Q * NT + RM * i + c] = (float)(v - (double)h);
            }
            if (i < H) {
                const double v = entry(H);
                const float h = (float)v;
                hi[H * NT + i] = h;
                lo[H * NT + i] = (float)(v - (double)h);
            }
            O.dg[e * NT + i] = entry(0);
        }
        zero_padding<NT>(e, lane, O.hi, O.lo);
    } else {
        // the triangle and its differences: lane j > 2t+1 receives the row
        // pair t's entries of column j (the product's exchange)
        double2 *Te = reinterpret_cast<double2 *>(O.K) + e * PAIRS;
        double *lw = reinterpret_cast<double *>(raw);
        const int t = i >> 1, o = 2 * (t * (NT - 3 - t) - 2) + (i & 1);
        bool fail = false;
        double diag = 0.0;
#pragma unroll
        for (int s = 0; s < H; ++s) {
            double own = i & 1 ? k[2 * s + 1] : k[2 * s];
            asm volatile("" : "+v"(own));   // a select per pair: not an indexed read of k, which would move it to memory
            diag = t == s ? own : diag;
            if (on && i <= 2 * s + 1) {
                Te[pf_tri_pair(s, i)] = make_double2(k[2 * s], k[2 * s + 1]);
            }
            if (s && on && i < 2 * s) {
                lw[o + 4 * s] = k[2 * s];
                lw[o + 4 * s + 2] = k[2 * s + 1];
            }
        }
        if (on) O.dg[e * NT + i] = diag;
        __syncthreads();
        const double2 *lr = reinterpret_cast<const double2 *>(raw);
        double dm = 0.0;
#pragma unroll
        for (int s = 0; s < H - 1; ++s) {
            if (!(on && i > 2 * s + 1)) continue;
            const double2 w = lr[s * (NT - 3 - s) + i - 2];
            const double d0 = __dsub_rn(k[2 * s], w.x), d1 = __dsub_rn(k[2 * s + 1], w.y);
            // with the check of the code below: the entry comes back exactly
            // (an infinite or undefined one does not; a sum that started at
            // +0 is never -0, so that equal entries are the same bits)
            fail |= __dadd_rn(w.x, d0) != k[2 * s] || __dadd_rn(w.y, d1) != k[2 * s + 1];
            k[2 * s] = d0;
            k[2 * s + 1] = d1;
            dm = fmax(dm, fmax(fabs(d0), fabs(d1)));
        }
        dm = wave_max(dm);
        dm = __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(dm)),
                              __builtin_amdgcn_readfirstlane(__double2loint(dm)));
        unsigned uh;
        double unit, inv;
        fail |= !tri_unit(dm, uh, unit, inv);
        unsigned *De = O.diff + e * LOW + i;
#pragma unroll
        for (int s = 0; s < H - 1; ++s) {
            if (!(on && i > 2 * s + 1)) continue;
            union { unsigned u; _Float16 h[2]; } c;
            c.h[0] = (_Float16)(float)(k[2 * s] * inv);
            c.h[1] = (_Float16)(float)(k[2 * s + 1] * inv);
            fail |= (double)c.h[0] * unit != k[2 * s] || (double)c.h[1] * unit != k[2 * s + 1];
            De[pf_tri_diff(NT, s, 0)] = c.u;
        }
        if (lane == 0) O.unit[e] = uh;
        if (fail) *O.bad = 1;
    }
}

// p123: kc{x,y,z} = sum_g d{x,y,z}_a d{x,y,z}_b det w; storkc = kx*kcx + ky*kcy + kz*kcz.
// Rows and columns enter every product alike, so K(a,b) = K(b,a) bit for bit
// and FP64 storage is the packed triangle without differences.
template <bool S32>
__global__ __launch_bounds__(64 * WAVES) void k_assemble_laplace8(
    const double *__restrict__ g_coord, const double *__restrict__ k_elem, double kx, double ky,
    double kz, double *__restrict__ T, float *__restrict__ hi, float *__restrict__ lo, double *__restrict__ dg,
    int nels)
{
    __shared__ ElemLds<8> lds[WAVES];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const long e = (long)blockIdx.x * WAVES + wave;
    const bool valid = e < nels;
    ElemLds<8> &L = lds[wave];
    element_geometry<8>(L, g_coord + (valid ? e : 0) * 24, lane, valid);
    if (!valid) return;
    const int a = lane & 7, b = lane >> 3;   // row a, column b
    double cx = 0.0, cy = 0.0, cz = 0.0;
#pragma unroll
    for (int g = 0; g < 8; ++g) {
        const double w = L.dw[g];
        cx += L.deriv[g][0][a] * L.deriv[g][0][b] * w;
        cy += L.deriv[g][1][a] * L.deriv[g][1][b] * w;
        cz += L.deriv[g][2][a] * L.deriv[g][2][b] * w;
    }
    const double s = k_elem ? k_elem[e] : 1.0;
    const double k = cx * (kx * s) + cy * (ky * s) + cz * (kz * s);
    if constexpr (S32) store_packed<8>(e, a, b, k, hi, lo, dg);
    else if (a <= (b | 1)) T[2 * (e * pf_tri_pairs(8) + pf_tri_pair(b >> 1, a)) + (b & 1)] = k;
}

// p124's element loop (src/programs/5th_ed/p124/p124.f90:73-86) on an
// 8-node brick: per Gauss point kc += MATMUL(MATMUL(TRANSPOSE(deriv),kay),
// deriv)*det*weights(i) with kay = diag(kx,ky,kz), pm += MATMUL(TRANSPOSE(
// funny),funny)*det*weights(i)*rho*cp with funny = SHAPE_FUN
// (new_library.f90:416-420); then storka = pm + kc*theta*dtim and storkb =
// pm - kc*(1-theta)*dtim.  prop(5,np_types) = kx, ky, kz, rho, cp per
// element type (READ_MATERIAL).  Every product and sum in the reference's
// order: MATMUL(TRANSPOSE(deriv),kay) has one nonzero term per entry (the
// others add exact zeros), the weights of SAMPLE are 1.  TRI: storka as the
// packed triangle with differences, an entry a lane, the mirrored one read
// across the wavefront (120^3 bricks, the whole call: whole matrices 2.76 ms,
// formed whole in chunks and packed from there 3.0, so 2.70).
template <bool TRI>
__global__ __launch_bounds__(64 * WAVES) void k_assemble_transient8(
    const double *__restrict__ g_coord, const double *__restrict__ prop, const int *__restrict__ etype,
    double theta, double dtim, as_out O, double *__restrict__ Kb, int nels)
{
    __shared__ ElemLds<8> lds[WAVES];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const long e = (long)blockIdx.x * WAVES + wave;
    const bool valid = e < nels;
    ElemLds<8> &L = lds[wave];
    element_geometry<8>(L, g_coord + (valid ? e : 0) * 24, lane, valid);
    if (!valid) return;
    const double *pr = prop + 5 * (long)(etype[e] - 1);
    const double kay[3] = {pr[0], pr[1], pr[2]}, rho = pr[3], cp = pr[4];
    const int a = lane & 7, b = lane >> 3;   // row a, column b
    // SHAPE_FUN, 8-node brick: node -> (xi, eta, zeta) factors, - = (1 - s),
    // + = (s + 1), each 0.125 * f_xi * f_eta * f_zeta
    constexpr int sx[8] = {-1, -1, 1, 1, -1, -1, 1, 1};
    constexpr int sy[8] = {-1, -1, -1, -1, 1, 1, 1, 1};
    constexpr int sz[8] = {-1, 1, 1, -1, -1, 1, 1, -1};
    constexpr double r3 = gauss_r3;
    double kc = 0.0, pm = 0.0;
#pragma unroll
    for (int g = 0; g < 8; ++g) {
        const double xi = gauss_sign[g][0] > 0 ? r3 : -r3, eta = gauss_sign[g][1] > 0 ? r3 : -r3,
                     zeta = gauss_sign[g][2] > 0 ? r3 : -r3;
        const double xim = 1.0 - xi, etam = 1.0 - eta, zetam = 1.0 - zeta;
        const double xip = xi + 1.0, etap = eta + 1.0, zetap = zeta + 1.0;
        const double fa = 0.125 * (sx[a] < 0 ? xim : xip) * (sy[a] < 0 ? etam : etap) * (sz[a] < 0 ? zetam : zetap);
        const double fb = 0.125 * (sx[b] < 0 ? xim : xip) * (sy[b] < 0 ? etam : etap) * (sz[b] < 0 ? zetam : zetap);
        const double det = L.dw[g];
        double t = 0.0;
#pragma unroll
        for (int m = 0; m < 3; ++m) t = t + (L.deriv[g][m][a] * kay[m]) * L.deriv[g][m][b];
        kc = kc + t * det * 1.0;
        pm = pm + fa * fb * det * 1.0 * rho * cp;
    }
    Kb[pf_idx_pair(e, 8, a, b)] = pm - kc * (1.0 - theta) * dtim;
    const double ka = pm + kc * theta * dtim;
    if constexpr (TRI) {
        const double up = __shfl(ka, 8 * a + b, 64);   // entry (b,a)
        const bool low = a > (b | 1);
        double dm = low ? fabs(__dsub_rn(ka, up)) : 0.0;
        dm = wave_max(dm);
        dm = __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(dm)),
                              __builtin_amdgcn_readfirstlane(__double2loint(dm)));
        unsigned uh;
        double unit, inv;
        bool fail = !tri_unit(dm, uh, unit, inv), code_fails = false;
        union { unsigned short u; _Float16 h; } c;
        c.h = tri_code(ka, up, inv, unit, code_fails);
        fail |= low && code_fails;
        const unsigned next = __shfl_down((unsigned)c.u, 8, 64);   // column b + 1
        if (!low) O.K[2 * (e * pf_tri_pairs(8) + pf_tri_pair(b >> 1, a)) + (b & 1)] = ka;
        else if (!(b & 1)) O.diff[e * pf_tri_diffs(8) + pf_tri_diff(8, b >> 1, a)] = c.u | next << 16;
        if (a == b) O.dg[e * 8 + a] = ka;
        if (lane == 0) O.unit[e] = uh;
        if (fail) *O.bad = 1;
    } else {
        O.K[pf_idx_pair(e, 8, a, b)] = ka;
    }
}

// hi = fl32(K), lo = fl32(K - hi) in the packed symmetric layout (upper
// triangle): hi + lo carries ~48 significant bits of K.
__global__ void k_split_fp32(const double *__restrict__ K, float *__restrict__ hi, float *__restrict__ lo,
                             int nt, long n)
{
    const long per = pf_sym_per(nt);
    const int Q4 = 4 * pf_sym_quads(nt), RF = pf_sym_rem(nt), H = nt / 2;
    for (long q = (long)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (long)gridDim.x * blockDim.x) {
        const long e = q / per;
        const int w = (int)(q - e * per);
        int i, d;
        if (w < Q4 * nt) {
            const int dq = w / (4 * nt), rem = w - dq * 4 * nt;
            i = rem >> 2;
            d = 4 * dq + (rem & 3);
        } else if (w < H * nt) {
            const int w2 = w - Q4 * nt;
            i = w2 / RF;
            d = Q4 + (w2 - i * RF);
        } else if (w < H * nt + H) {
            i = w - H * nt;
            d = H;
        } else {                        // padding
            hi[q] = 0.0f;
            lo[q] = 0.0f;
            continue;
        }
        int j = i + d;
        if (j >= nt) j -= nt;
        const double k = K[pf_idx_pair(e, nt, i < j ? i : j, i < j ? j : i)];
        const float h = (float)k;
        hi[q] = h;
        lo[q] = (float)(k - (double)h);
    }
}

// storkm_pp chunk (column-major, elements e0..e0+nel-1) -> FP64 pair layout.
__global__ void k_from_colmajor(const double *__restrict__ src, double *__restrict__ K, int nt, long e0, long nel)
{
    const long nn = (long)nt * nt, n = nel * nn;
    for (long q = (long)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (long)gridDim.x * blockDim.x) {
        const long el = q / nn, w = q - el * nn;
        const int j = (int)(w / nt), i = (int)(w - (long)j * nt);
        K[pf_idx_pair(e0 + el, nt, i, j)] = src[q];
    }
}

// FP64 matrices (column-major) -> packed triangle.  One lane
// group per element (lane = row), the whole matrix in LDS; every entry below
// the diagonal is reconstructed as the product will and compared (with T null
// only that).  Bound by the reads of src, which a bounded chunk leaves in the
// last-level cache.
template <int NT>
__global__ __launch_bounds__(64) void k_tri_pack(const double *__restrict__ src, double *__restrict__ T,
                                                unsigned *__restrict__ diff, unsigned *__restrict__ unit, long e0,
                                                long nel, int *__restrict__ bad)
{
    constexpr int W = NT > 32 ? 64 : (NT > 16 ? 32 : 8), EPW = 64 / W, H = NT / 2, PITCH = NT + 1;
    __shared__ double m[EPW][NT * PITCH];
    const int lane = threadIdx.x & 63, sub = lane / W, i = lane % W;
    const long el = (long)blockIdx.x * EPW + sub;
    const bool on = el < nel && i < NT;
    double *M = m[sub];
    const double *S = src + (el < nel ? el : 0) * (long)(NT * NT);
    if (on) {
#pragma unroll
        for (int s = 0; s < H; ++s) {
            M[i * PITCH + 2 * s] = S[2 * s * NT + i];
            M[i * PITCH + 2 * s + 1] = S[(2 * s + 1) * NT + i];
        }
    }
    __syncthreads();
    // the largest difference of the element
    double dm = 0.0;
    if (on)
        for (int j = 0; j < (i & ~1); ++j) dm = fmax(dm, fabs(__dsub_rn(M[i * PITCH + j], M[j * PITCH + i])));
    for (int off = W / 2; off > 0; off >>= 1) dm = fmax(dm, __shfl_xor(dm, off, 64));
    unsigned uh;
    double un, inv;
    bool fail = !tri_unit(dm, uh, un, inv) && on;
    const long e = e0 + el;
    if (on) {
        double2 *Te = reinterpret_cast<double2 *>(T) + e * pf_tri_pairs(NT);
        unsigned *De = diff + e * pf_tri_diffs(NT);
        for (int s = 0; s < H; ++s) {
            const double a = M[i * PITCH + 2 * s], b = M[i * PITCH + 2 * s + 1];
            if (i <= 2 * s + 1) {
                if (T) Te[pf_tri_pair(s, i)] = make_double2(a, b);
                continue;
            }
            const double ua = M[2 * s * PITCH + i], ub = M[(2 * s + 1) * PITCH + i];
            union { unsigned u; _Float16 h[2]; } w;
            w.h[0] = tri_code(a, ua, inv, un, fail);
            w.h[1] = tri_code(b, ub, inv, un, fail);
            if (T) De[pf_tri_diff(NT, s, i)] = w.u;
        }
        if (T && i == 0) unit[e] = uh;
    }
    if (fail) *bad = 1;
}

// Elements 0 .. nel - 1 of the packed triangle -> column pairs.
__global__ void k_tri_unpack(pf_f64_view V, double *__restrict__ K, int nt, long nel)
{
    const long nn = (long)nt * nt, n = nel * nn;
    for (long q = (long)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (long)gridDim.x * blockDim.x) {
        const long el = q / nn, w = q - el * nn;
        const int j = (int)(w / nt), i = (int)(w - (long)j * nt);
        K[pf_idx_pair(el, nt, i, j)] = pf_f64_entry(V, el, nt, i, j);
    }
}

// internal layout -> storkm_pp chunk (FP64, or packed symmetric hi + lo).
__global__ void k_to_colmajor(pf_f64_view V, const float *__restrict__ hi, const float *__restrict__ lo,
                              double *__restrict__ dst, int nt, long e0, long nel)
{
    const long nn = (long)nt * nt, n = nel * nn;
    for (long q = (long)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (long)gridDim.x * blockDim.x) {
        const long el = q / nn, w = q - el * nn;
        const int j = (int)(w / nt), i = (int)(w - (long)j * nt);
        if (V.K || V.T) {
            dst[q] = pf_f64_entry(V, e0 + el, nt, i, j);
        } else {
            const long t = pf_idx_sym_ij(e0 + el, nt, i, j);
            dst[q] = (double)hi[t] + (double)lo[t];
        }
    }
}

// Assembled diagonal: diag(q) = sum over the slots of q, ascending element,
// of storkm(i,i,e) (p121.f90:65-69 then SCATTER).  diag has a leading 0 slot.
__global__ void k_diag(const int *__restrict__ ptr, const int *__restrict__ slot, pf_f64_view V, int ntot,
                       double *__restrict__ diag, int neq)
{
    for (int q = blockIdx.x * blockDim.x + threadIdx.x; q < neq; q += gridDim.x * blockDim.x) {
        double s = 0.0;
        for (int k = ptr[q]; k < ptr[q + 1]; ++k) {
            const long sl = slot[k];
            const long e = sl / ntot;
            const int i = (int)(sl - e * ntot);
            s = __dadd_rn(s, pf_f64_entry(V, e, ntot, i, i));
        }
        diag[q + 1] = s;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) diag[0] = 0.0;
}

// The same diagonal from the FP64 element diagonals dg(ntot,nels) that the
// FP32-storage assembly writes.
__global__ void k_diag_elem(const int *__restrict__ ptr, const int *__restrict__ slot,
                            const double *__restrict__ dg, double *__restrict__ diag, int neq)
{
    for (int q = blockIdx.x * blockDim.x + threadIdx.x; q < neq; q += gridDim.x * blockDim.x) {
        double s = 0.0;
        for (int k = ptr[q]; k < ptr[q + 1]; ++k) s = __dadd_rn(s, dg[slot[k]]);
        diag[q + 1] = s;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) diag[0] = 0.0;
}

}  // namespace

// FP32 storage writes K32hi/K32lo, FP64 storage the triangle (*bad set where
// it does not hold), both with the element diagonals in dg (ntot*nels
// doubles); FP64 storage without a triangle writes K64.
int pf_launch_assemble_elastic(pf_ctx *c, double v2, double vv, double den, double e, const double *e_elem,
                               double *dg, int *bad)
{
    const bool s32 = c->store == PF_STORE_FP32, tri = !s32 && c->T64;
    if (s32 ? !c->K32hi || !c->K32lo || !dg : tri ? !c->T64d || !c->T64u || !bad || !dg : !c->K64) return PF_ERR_STATE;
    const as_out O{tri ? c->T64 : c->K64, c->T64d, c->T64u, bad, c->K32hi, c->K32lo, dg};
    const dim3 grid(c->nels), blk(64);
#define PF_AS(NOD, MODE)                                                                                           \
    hipLaunchKernelGGL((k_assemble_elastic<NOD, MODE>), grid, blk, 0, c->stream, c->g_coord, e_elem, v2, vv, den, e, O)
    if (c->nod == 20) {
        if (s32) PF_AS(20, AS_PACK32);
        else if (tri) PF_AS(20, AS_TRI);
        else PF_AS(20, AS_PAIRS);
    } else if (c->nod == 8) {
        if (s32) PF_AS(8, AS_PACK32);
        else if (tri) PF_AS(8, AS_TRI);
        else PF_AS(8, AS_PAIRS);
    } else {
        return PF_ERR_ARG;
    }
#undef PF_AS
    PF_HIP(hipGetLastError());
    return PF_OK;
}

int pf_launch_assemble_laplace(pf_ctx *c, double kx, double ky, double kz, const double *k_elem, double *dg)
{
    if (c->nod != 8) return PF_ERR_ARG;
    const int grid = (c->nels + WAVES - 1) / WAVES;
    if (c->store == PF_STORE_FP32) {
        if (!c->K32hi || !c->K32lo || !dg) return PF_ERR_STATE;
        hipLaunchKernelGGL(k_assemble_laplace8<true>, dim3(grid), dim3(64 * WAVES), 0, c->stream, c->g_coord,
                           k_elem, kx, ky, kz, (double *)nullptr, c->K32hi, c->K32lo, dg, c->nels);
    } else {
        if (!c->T64) return PF_ERR_STATE;
        hipLaunchKernelGGL(k_assemble_laplace8<false>, dim3(grid), dim3(64 * WAVES), 0, c->stream, c->g_coord,
                           k_elem, kx, ky, kz, c->T64, (float *)nullptr, (float *)nullptr, (double *)nullptr,
                           c->nels);
    }
    PF_HIP(hipGetLastError());
    return PF_OK;
}

template <int NT>
static void launch_tri_pack(pf_ctx *c, const double *src, long e0, long nel, int *bad)
{
    constexpr int EPW = NT > 32 ? 1 : (NT > 16 ? 2 : 8);
    hipLaunchKernelGGL(k_tri_pack<NT>, dim3((unsigned)((nel + EPW - 1) / EPW)), dim3(64), 0, c->stream, src, c->T64,
                       c->T64d, c->T64u, e0, nel, bad);
}

int pf_launch_tri_pack(pf_ctx *c, const double *src, long e0, long nel, int *bad)
{
    if (c->T64 && (!c->T64d || !c->T64u)) return PF_ERR_STATE;
    switch (c->ntot) {
    case 60: launch_tri_pack<60>(c, src, e0, nel, bad); break;
    case 24: launch_tri_pack<24>(c, src, e0, nel, bad); break;
    case 8: launch_tri_pack<8>(c, src, e0, nel, bad); break;
    default: return PF_ERR_ARG;
    }
    PF_HIP(hipGetLastError());
    return PF_OK;
}

int pf_launch_tri_unpack(pf_ctx *c, double *K, long nel)
{
    if (!c->T64) return PF_ERR_STATE;
    hipLaunchKernelGGL(k_tri_unpack, dim3(8192), dim3(256), 0, c->stream, pf_f64(c), K, c->ntot, nel);
    PF_HIP(hipGetLastError());
    return PF_OK;
}

int pf_launch_diag_elem(pf_ctx *c, const double *dg, double *diag)
{
    const int grid = (c->neq + 255) / 256 < 8192 ? (c->neq + 255) / 256 : 8192;
    hipLaunchKernelGGL(k_diag_elem, dim3(grid), dim3(256), 0, c->stream, c->csr_ptr, c->csr_slot, dg, diag, c->neq);
    PF_HIP(hipGetLastError());
    return PF_OK;
}

int pf_launch_assemble_transient(pf_ctx *c, double theta, double dtim, const double *prop, const int *etype,
                                 int *bad)
{
    if (c->nod != 8) return PF_ERR_ARG;
    if (!c->K64b || (c->T64 ? !c->T64d || !c->T64u || !bad : !c->K64)) return PF_ERR_STATE;
    const as_out O{c->T64 ? c->T64 : c->K64, c->T64d, c->T64u, bad, nullptr, nullptr, c->utemp};
    const dim3 grid((c->nels + WAVES - 1) / WAVES), blk(64 * WAVES);
    if (c->T64)
        hipLaunchKernelGGL(k_assemble_transient8<true>, grid, blk, 0, c->stream, c->g_coord, prop, etype, theta, dtim, O,
                           c->K64b, c->nels);
    else
        hipLaunchKernelGGL(k_assemble_transient8<false>, grid, blk, 0, c->stream, c->g_coord, prop, etype, theta, dtim,
                           O, c->K64b, c->nels);
    PF_HIP(hipGetLastError());
    return PF_OK;
}

int pf_launch_split_fp32(pf_ctx *c)
{
    const long n = pf_sym_per(c->ntot) * c->nels;
    hipLaunchKernelGGL(k_split_fp32, dim3(8192), dim3(256), 0, c->stream, c->K64, c->K32hi, c->K32lo, c->ntot, n);
    PF_HIP(hipGetLastError());
    return PF_OK;
}

int pf_launch_from_colmajor(pf_ctx *c, const double *src, long e0, long nel)
{
    hipLaunchKernelGGL(k_from_colmajor, dim3(8192), dim3(256), 0, c->stream, src, c->K64, c->ntot, e0, nel);
    PF_HIP(hipGetLastError());
    return PF_OK;
}

int pf_launch_to_colmajor(pf_ctx *c, double *dst, long e0, long nel)
{
    hipLaunchKernelGGL(k_to_colmajor, dim3(8192), dim3(256), 0, c->stream, pf_f64(c), c->K32hi, c->K32lo, dst,
                       c->ntot, e0, nel);
    PF_HIP(hipGetLastError());
    return PF_OK;
}

int pf_launch_diag(pf_ctx *c, double *diag)
{
    const int grid = (c->neq + 255) / 256 < 8192 ? (c->neq + 255) / 256 : 8192;
    hipLaunchKernelGGL(k_diag, dim3(grid), dim3(256), 0, c->stream, c->csr_ptr, c->csr_slot, pf_f64(c), c->ntot,
                       diag, c->neq);
    PF_HIP(hipGetLastError());
    return PF_OK;
}

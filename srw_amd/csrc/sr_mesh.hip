// sr_mesh.hip - the method-0 SR integral of a transverse mesh as a matrix
// product on the matrix cores (gfx950).
//
// The phase of the reference's integrand (cpp/src/core/srradint.h:884-919) at
// mesh point (x, z) and integration point s is, in revolutions,
//   k [Q(s) + (x - X(s))^2 / (y - s)]  +  k (z - Z(s))^2 / (y - s),
// a part of (x, s) plus a part of (z, s), and each amplitude depends on one of
// the two coordinates.  With F = exp(2 pi i (first part)), G = exp(2 pi i
// (second part)), F' = b (Px - x) F and G' = b (Pz - z) G the two components
//   Ex(x, z) = sum_s F'(x, s) G(z, s),   Ez(x, z) = sum_s F(x, s) G'(z, s)
// are complex matrix products over s: (nx + nz) ns phasors and 8 real
// multiply-adds per evaluation replace a phase, a sine and a cosine each.
#include "srw_sr_dev.h"

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float float2v __attribute__((ext_vector_type(2)));
typedef float float16v __attribute__((ext_vector_type(16)));
typedef unsigned uint4v __attribute__((ext_vector_type(4)));

#define MESH_STAGE 16                                 // integration points per LDS stage (one MFMA's k)
#define MESH_FLUSH (SRWD_MESH_UNIT / MESH_STAGE)      // stages between FP64 flushes
#define MESH_PLANE (2 * 64)                           // 16-byte words of one plane: 2 blocks of 32 rows x 2 k-groups x 32
#define MESH_BUF (16 * MESH_PLANE)

typedef const __attribute__((address_space(4))) srwd_mrec* mrec_ptr;

__device__ __forceinline__ mrec_ptr mesh_rec_ptr(const srwd_mrec* p)
{
    const unsigned long long v = (unsigned long long)p;
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)v);
    const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(v >> 32));
    return (mrec_ptr)(((unsigned long long)hi << 32) | lo);
}

// Two floats as the sum of two FP16 pairs: v = hi + lo to about 22 bits.
__device__ __forceinline__ void split2(float a, float b, unsigned& hi, unsigned& lo)
{
    const half2v h = __builtin_convertvector((float2v){a, b}, half2v);
    const half2v l = __builtin_convertvector((float2v){a - (float)h.x, b - (float)h.y}, half2v);
    hi = __builtin_bit_cast(unsigned, h);
    lo = __builtin_bit_cast(unsigned, l);
}

// The phasor and the weighted phasor of one coordinate at 8 integration
// points R[0..7], as 8 planes (phasor re hi, re lo, im hi, im lo; weighted
// the same) of 8 FP16 values.  X = 1: the x side (carries Q), 0: the z side.
template <int X>
__device__ __forceinline__ void mesh_gen(double r0, double kap, float scale, mrec_ptr R, uint4v* dst)
{
    unsigned o[8][4];
    const float nr = -(float)r0;
#pragma unroll
    for (int p = 0; p < 4; p++) {
        float cs[2], sn[2], wc[2], ws[2];
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int i = 2 * p + u;
            const double d = r0 - (X ? R[i].X : R[i].Z);
            const double q = d * d;
            const double t = kap * (X ? fma(q, R[i].inv, R[i].sQ) : q * R[i].inv);
            const float f = (float)(t - rint(t));
            cs[u] = __builtin_amdgcn_cosf(f);
            sn[u] = __builtin_amdgcn_sinf(f);
            const float a = scale * fmaf(R[i].b, nr, X ? R[i].bPx : R[i].bPz);
            wc[u] = a * cs[u];
            ws[u] = a * sn[u];
        }
        split2(cs[0], cs[1], o[0][p], o[1][p]);
        split2(sn[0], sn[1], o[2][p], o[3][p]);
        split2(wc[0], wc[1], o[4][p], o[5][p]);
        split2(ws[0], ws[1], o[6][p], o[7][p]);
    }
#pragma unroll
    for (int k = 0; k < 8; k++) dst[k * MESH_PLANE] = (uint4v){o[k][0], o[k][1], o[k][2], o[k][3]};
}

__device__ __forceinline__ float16v mfma(uint4v a, uint4v b, float16v c)
{
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, a), __builtin_bit_cast(half8, b), c, 0, 0,
                                                  0);
}

// One complex product: re += Ar Br - Ai Bi, im += Ar Bi + Ai Br, each factor
// as hi + lo (the lo lo part, 2^-22 of a term, is left out).  A points to the
// planes re hi, re lo, im hi, im lo of the rows, B to those of the columns.
__device__ __forceinline__ void mesh_cmac(const uint4v* A, const uint4v* B, float16v& re, float16v& im)
{
    const uint4v arh = A[0], arl = A[MESH_PLANE], aih = A[2 * MESH_PLANE], ail = A[3 * MESH_PLANE];
    const uint4v brh = B[0], brl = B[MESH_PLANE], bih = B[2 * MESH_PLANE], bil = B[3 * MESH_PLANE];
    const uint4v nih = aih ^ 0x80008000u, nil = ail ^ 0x80008000u;
    re = mfma(arh, brh, re);
    im = mfma(arh, bih, im);
    re = mfma(nih, bih, re);
    im = mfma(aih, brh, im);
    re = mfma(arl, brh, re);
    im = mfma(arl, bih, im);
    re = mfma(nil, bih, re);
    im = mfma(ail, brh, im);
    re = mfma(arh, brl, re);
    im = mfma(arh, bil, im);
    re = mfma(nih, bil, re);
    im = mfma(aih, brl, im);
}

__global__ void __launch_bounds__(256, 2) k_sr_mesh(const srwd_item* __restrict__ items, const int2* __restrict__ tiles,
                                                    const srwd_trj_info* __restrict__ info,
                                                    const srwd_mrec* __restrict__ rec, long long ldM,
                                                    const double* __restrict__ cond, int nSplit, long long nPointsPad,
                                                    double* __restrict__ part)
{
    __shared__ uint4v lds[2 * MESH_BUF];
    const int2 tl = tiles[blockIdx.x];
    const srwd_item& IT = items[tl.x];
    const int nxc = IT.nxc, nzr = IT.npts / nxc;
    const int nTx = (nxc + SRWD_MESH_TILE - 1) / SRWD_MESH_TILE;
    const int tx = (tl.y % nTx) * SRWD_MESH_TILE, tz = (tl.y / nTx) * SRWD_MESH_TILE;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // amplitude scales (powers of two): the largest weighted phasor is kept
    // below 2^12, well inside FP16
    const double* cd = cond + SRWD_COND * IT.traj;
    const double xm = fmax(fabs(IT.xStart), fabs(IT.xStart + (IT.nx - 1) * IT.xStep));
    const double zm = fmax(fabs(IT.zStart), fabs(IT.zStart + (IT.nz - 1) * IT.zStep));
    const double ax = cd[5] * xm + cd[6], az = cd[5] * zm + cd[7];
    const int ex = ax > 0. ? 11 - ilogb(ax) : 0, ez = az > 0. ? 11 - ilogb(az) : 0;
    // this block's stages
    const int nUnit = (int)((info[IT.traj].nInt + SRWD_MESH_UNIT - 1) / SRWD_MESH_UNIT);
    const int u0 = (int)((long long)nUnit * blockIdx.y / nSplit), u1 = (int)((long long)nUnit * (blockIdx.y + 1) / nSplit);
    const srwd_mrec* R = rec + (long long)IT.traj * ldM;
    // phasors: waves 0, 1 the x side, waves 2, 3 the z side, one row of the
    // tile per lane; a wave takes 8 of the stage's 16 integration points, so
    // the trajectory data are uniform (scalar loads)
    const int side = w >> 1, sg = w & 1;
    const double kap = SRWD_KPH(IT.eph) * (0.5 / M_PI);
    const int row = min(side ? tz + lane : tx + lane, side ? nzr - 1 : nxc - 1);
    const double crd = side ? IT.zStart + (IT.iz0 + row) * IT.zStep : IT.xStart + row * IT.xStep;
    const float sc = (float)ldexp(1., side ? ez : ex);
    uint4v* wr = lds + side * 8 * MESH_PLANE + (lane >> 5) * 64 + sg * 32 + (lane & 31);
    auto gen = [&](int stage, int buf) {
        mrec_ptr r = mesh_rec_ptr(R + (long long)stage * MESH_STAGE + sg * 8);
        if (side) mesh_gen<0>(crd, kap, sc, r, wr + buf * MESH_BUF);
        else mesh_gen<1>(crd, kap, sc, r, wr + buf * MESH_BUF);
    };
    // products: wave (wz, wx) takes 32 z rows (A) x 32 x columns (B)
    const int wx = w & 1, wz = w >> 1;
    const bool live = tx + 32 * wx < nxc && tz + 32 * wz < nzr;
    const uint4v* rdX = lds + wx * 64 + lane;
    const uint4v* rdZ = lds + 8 * MESH_PLANE + wz * 64 + lane;
    float16v xr, xi, zr, zi;
    double o[4][16];
#pragma unroll
    for (int i = 0; i < 16; i++) o[0][i] = o[1][i] = o[2][i] = o[3][i] = 0.;
    const int s0 = u0 * MESH_FLUSH, s1 = u1 * MESH_FLUSH;
    if (s0 < s1) gen(s0, 0);
    __syncthreads();
    for (int s = s0; s < s1; s += MESH_FLUSH) {
        xr = xi = zr = zi = (float16v)0.f;
#pragma unroll 1
        for (int k = 0; k < MESH_FLUSH; k++) {
            const int buf = k & 1;
            if (live) {
                mesh_cmac(rdZ + buf * MESH_BUF, rdX + buf * MESH_BUF + 4 * MESH_PLANE, xr, xi);
                mesh_cmac(rdZ + buf * MESH_BUF + 4 * MESH_PLANE, rdX + buf * MESH_BUF, zr, zi);
            }
            if (s + k + 1 < s1) gen(s + k + 1, buf ^ 1);
            __syncthreads();
        }
        if (live) {
#pragma unroll
            for (int i = 0; i < 16; i++) {
                o[0][i] += (double)xr[i]; o[1][i] += (double)xi[i];
                o[2][i] += (double)zr[i]; o[3][i] += (double)zi[i];
            }
        }
    }
    if (!live) return;
    const double ux = ldexp(1., -ex), uz = ldexp(1., -ez);
    const int ix = tx + 32 * wx + (lane & 31);
    if (ix >= nxc) return;
    double* P = part + ((long long)blockIdx.y * nPointsPad + IT.pointBase) * 4;
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const int iz = tz + 32 * wz + (i & 3) + 8 * (i >> 2) + 4 * (lane >> 5);
        if (iz >= nzr) continue;
        double2* d = (double2*)(P + 4 * ((long long)iz * nxc + ix));
        d[0] = make_double2(o[0][i] * ux, o[1][i] * ux);
        d[1] = make_double2(o[2][i] * uz, o[3][i] * uz);
    }
}

extern "C" int srwd_launch_sr_mesh(const srwd_item* dItems, const int2* dTiles, int nTiles, const srwd_trj_info* dInfo,
                                   const srwd_mrec* dRec, long long ldM, const double* dCond, int nSplit,
                                   long long nPointsPad, double* dPart, hipStream_t st)
{
    if (nTiles <= 0) return 0;
    hipLaunchKernelGGL(k_sr_mesh, dim3(nTiles, nSplit), dim3(256), 0, st, dItems, dTiles, dInfo, dRec, ldM, dCond, nSplit,
                       nPointsPad, dPart);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

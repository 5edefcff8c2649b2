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
//
// What bounds it: the matrix instructions (24 of 32x32x16 per 16 points and
// 32 x 32 places, 48 FP16 flops an evaluation) and the vector work of the
// phasors, which share a SIMD's issue: with either left out a launch took 5.2
// of 8.1 ms (64 electrons on 512 x 512), so about half of the matrix time hides
// behind the vector work.  512 x 512 points of 256 electrons: 36 ms, 0.9 of
// 1.85 PFLOP/s that a plain loop of these instructions reaches here; one lane
// per point with vector FMAs (k_sr_integral) took 176 ms.
// * 64 x 64 tile: a phasor serves 64 points, and the two buffers of a stage
//   (64 KB of LDS) leave two workgroups a CU, one's phasors beside the other's
//   products.
// * 16 points a stage: one instruction's k.  The products of hi and lo parts
//   are summed small ones first.
// * FP32 sums flushed to FP64 every 32 points (SRWD_MESH_UNIT): at 64 the
//   kernel was 3 to 11 % faster and fields far below their peak carried more
//   error than one lane per point gives; at 128 single points failed 1e-4.
// * s_setprio around the products: 3 %.
#include "srw_sr_dev.h"

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float float2v __attribute__((ext_vector_type(2)));
typedef float float16v __attribute__((ext_vector_type(16)));
typedef int int16v __attribute__((ext_vector_type(16)));
typedef unsigned uint4v __attribute__((ext_vector_type(4)));

#define MESH_STAGE 16                                 // integration points per LDS stage (one MFMA's k): 2 groups
#define MESH_FLUSH (SRWD_MESH_UNIT / MESH_STAGE)      // stages between FP64 flushes
#define MESH_PLANE (2 * 64)                           // 16-byte words of one plane: 2 blocks of 32 rows x 2 k-groups x 32
#define MESH_BUF (16 * MESH_PLANE)

// A group of integration points in scalar registers.
struct mesh_grp {
    int16v v[3];
    __device__ __forceinline__ double f64(int k) const
    {
        const unsigned long long lo = (unsigned)v[0][2 * k], hi = (unsigned)v[0][2 * k + 1];
        return __builtin_bit_cast(double, lo | (hi << 32));
    }
    // field k (0 dq, 1 du, 2 di, 3 b, 4 p) of point i
    __device__ __forceinline__ float f32(int k, int i) const
    {
        const int at = 8 + 8 * k + i;
        return __builtin_bit_cast(float, (int)v[at >> 4][at & 15]);
    }
};

// p is the same for the whole wave.
__device__ __forceinline__ mesh_grp mesh_load(const srwd_mrec* p)
{
    const unsigned long long a = (unsigned long long)p;
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)a);
    const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(a >> 32));
    const __attribute__((address_space(4))) int16v* q =
        (const __attribute__((address_space(4))) int16v*)(((unsigned long long)hi << 32) | lo);
    mesh_grp r;
#pragma unroll
    for (int k = 0; k < 3; k++) r.v[k] = q[k];
    return r;
}

// FP16 pairs hi + lo of a pair of floats (about 22 bits each): split2 of a
// and b, splitp of the products a*u and b*v.  The mixed FMAs round once, into
// the low or the high half of the result.
__device__ __forceinline__ void split2(float a, float b, unsigned& hi, unsigned& lo)
{
    hi = __builtin_bit_cast(unsigned, __builtin_convertvector((float2v){a, b}, half2v));
    asm("v_fma_mixlo_f16 %0, %1, 1.0, -%2 op_sel:[0,0,0] op_sel_hi:[0,0,1]" : "=v"(lo) : "v"(a), "v"(hi));
    asm("v_fma_mixhi_f16 %0, %1, 1.0, -%2 op_sel:[0,0,1] op_sel_hi:[0,0,1]" : "+v"(lo) : "v"(b), "v"(hi));
}

__device__ __forceinline__ void splitp(float a, float u, float b, float v, unsigned& hi, unsigned& lo)
{
    asm("v_fma_mixlo_f16 %0, %1, %2, 0" : "=v"(hi) : "v"(a), "v"(u));
    asm("v_fma_mixhi_f16 %0, %1, %2, 0" : "+v"(hi) : "v"(b), "v"(v));
    asm("v_fma_mixlo_f16 %0, %1, %2, -%3 op_sel:[0,0,0] op_sel_hi:[0,0,1]" : "=v"(lo) : "v"(a), "v"(u), "v"(hi));
    asm("v_fma_mixhi_f16 %0, %1, %2, -%3 op_sel:[0,0,1] op_sel_hi:[0,0,1]" : "+v"(lo) : "v"(b), "v"(v), "v"(hi));
}

// The row of a tile that a lane forms phasors of: its coordinate, k in
// revolutions per metre, and the factors of the phase increments.
struct mesh_row {
    double r, k;
    float x, xl, kf, beta, alpha;   // x + xl = r
};

// The phasor and the weighted phasor of one row at the 8 integration points
// of G, as 8 planes (phasor re hi, re lo, im hi, im lo; weighted the same) of
// 8 FP16 values.  The phase at the reference point is formed and reduced in FP64;
// the other points add FP32 increments (srwd_mesh_turns).
__device__ __forceinline__ void mesh_gen(const mesh_row& W, const mesh_grp& G, uint4v* dst)
{
    unsigned o[8][4];
    const double d = W.r - G.f64(0);
    const double tc = W.k * fma(d * G.f64(1), d, G.f64(2));
    const double tr = tc - rint(tc);
    const float t0 = (float)tr, t1 = (float)(tr - t0);
#pragma unroll
    for (int p = 0; p < 4; p++) {
        float cs[2], sn[2], a[2];
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int i = 2 * p + u;
            const float t = t0 + fmaf(W.alpha, G.f32(2, i), fmaf(W.beta, G.f32(1, i), fmaf(W.kf, G.f32(0, i), t1)));
            cs[u] = __builtin_amdgcn_cosf(t);
            sn[u] = __builtin_amdgcn_sinf(t);
            a[u] = ((G.f32(4, i) - W.x) - W.xl) * G.f32(3, i);
        }
        split2(cs[0], cs[1], o[0][p], o[1][p]);
        split2(sn[0], sn[1], o[2][p], o[3][p]);
        splitp(a[0], cs[0], a[1], cs[1], o[4][p], o[5][p]);
        splitp(a[0], sn[0], a[1], sn[1], o[6][p], o[7][p]);
    }
#pragma unroll
    for (int k = 0; k < 8; k++) dst[k * MESH_PLANE] = (uint4v){o[k][0], o[k][1], o[k][2], o[k][3]};
}

__device__ __forceinline__ float16v mfma(uint4v a, uint4v b, float16v c)
{
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, a), __builtin_bit_cast(half8, b), c, 0, 0,
                                                  0);
}

// The four planes (re hi, re lo, im hi, im lo) of one side as MFMA operands.
struct mesh_op {
    uint4v rh, rl, ih, il;
    __device__ __forceinline__ mesh_op(const uint4v* p)
        : rh(p[0]), rl(p[MESH_PLANE]), ih(p[2 * MESH_PLANE]), il(p[3 * MESH_PLANE]) {}
};

// One complex product: re += Ar Br - Ai Bi, im += Ar Bi + Ai Br, each factor
// as hi + lo (the lo lo part, 2^-22 of a term, is left out).
__device__ __forceinline__ void mesh_cmac(const mesh_op& A, const mesh_op& B, float16v& re, float16v& im)
{
    const uint4v nh = A.ih ^ 0x80008000u, nl = A.il ^ 0x80008000u;
    re = mfma(A.rl, B.rh, re);
    im = mfma(A.rl, B.ih, im);
    re = mfma(nl, B.ih, re);
    im = mfma(A.il, B.rh, im);
    re = mfma(A.rh, B.rl, re);
    im = mfma(A.rh, B.il, im);
    re = mfma(nh, B.il, re);
    im = mfma(A.ih, B.rl, im);
    re = mfma(A.rh, B.rh, re);
    im = mfma(A.rh, B.ih, im);
    re = mfma(nh, B.ih, re);
    im = mfma(A.ih, B.rh, im);
}

__global__ void __launch_bounds__(256, 2) k_sr_mesh(const srwd_item* __restrict__ items, const int2* __restrict__ tiles, int ntU,
                                                    const srwd_trj_info* __restrict__ info,
                                                    const srwd_mrec* __restrict__ rec, long long ldM,
                                                    const double* __restrict__ scale, int nSplit, long long nPointsPad,
                                                    double* __restrict__ part)
{
    __shared__ uint4v lds[2 * MESH_BUF];
    const int2 tl = tiles ? tiles[blockIdx.x] : make_int2(blockIdx.x / ntU, blockIdx.x % ntU);
    const srwd_item& IT = items[tl.x];
    const int nxc = IT.nxc, nzr = IT.npts / nxc;
    const int nTx = (nxc + SRWD_MESH_TILE - 1) / SRWD_MESH_TILE;
    const int tx = (tl.y % nTx) * SRWD_MESH_TILE, tz = (tl.y / nTx) * SRWD_MESH_TILE;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // this block's stages
    const int nUnit = (int)((info[IT.traj].nInt + SRWD_MESH_UNIT - 1) / SRWD_MESH_UNIT);
    const int u0 = (int)((long long)nUnit * blockIdx.y / nSplit), u1 = (int)((long long)nUnit * (blockIdx.y + 1) / nSplit);
    // phasors: waves 0, 1 the x side, waves 2, 3 the z side, one row of the
    // tile per lane; a wave takes 8 of the stage's 16 integration points, so
    // the trajectory data are uniform (scalar loads)
    const int side = w >> 1, sg = w & 1;
    const int row = min(side ? tz + lane : tx + lane, side ? nzr - 1 : nxc - 1);
    mesh_row W;
    W.r = side ? IT.zStart + (IT.iz0 + row) * IT.zStep : IT.xStart + row * IT.xStep;
    W.k = SRWD_KPH(IT.eph) * (0.5 / M_PI);
    W.x = (float)W.r; W.xl = (float)(W.r - W.x); W.kf = (float)W.k; W.beta = (float)(-2. * W.k * W.r); W.alpha = (float)(W.k * W.r * W.r);
    uint4v* wr = lds + side * 8 * MESH_PLANE + (lane >> 5) * 64 + sg * 32 + (lane & 31);
    const srwd_mrec* R = rec + (2LL * IT.traj + side) * ldM + sg;
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
    mesh_gen(W, mesh_load(R + 2LL * s0), wr);
    __syncthreads();
    if (live) {
        for (int s = s0; s < s1; s += MESH_FLUSH) {
            xr = xi = zr = zi = (float16v)0.f;
#pragma unroll
            for (int k = 0; k < MESH_FLUSH; k++) {
                const int buf = (k & 1) * MESH_BUF;
                const mesh_op zg(rdZ + buf), xw(rdX + buf + 4 * MESH_PLANE);
                // LDS reads and scalar loads share a counter that the latter
                // leave out of order: the records of the next stage are asked
                // for once the operands are there, and arrive behind the MFMAs
                __builtin_amdgcn_s_waitcnt(0xC07F);
                const mesh_grp next = mesh_load(R + 2LL * (s + k + 1));
                __builtin_amdgcn_sched_barrier(0);
                __builtin_amdgcn_s_setprio(1);
                mesh_cmac(zg, xw, xr, xi);
                const mesh_op zw(rdZ + buf + 4 * MESH_PLANE), xg(rdX + buf);
                mesh_cmac(zw, xg, zr, zi);
                __builtin_amdgcn_sched_barrier(0);
                __builtin_amdgcn_s_setprio(0);
                mesh_gen(W, next, wr + (MESH_BUF - buf));
                __syncthreads();
            }
#pragma unroll
            for (int i = 0; i < 16; i++) {
                o[0][i] += (double)xr[i]; o[1][i] += (double)xi[i];
                o[2][i] += (double)zr[i]; o[3][i] += (double)zi[i];
            }
        }
    } else {
        // nothing of the tile to sum here: the phasors only
        for (int s = s0; s < s1; s++) {
            mesh_gen(W, mesh_load(R + 2LL * (s + 1)), wr + (((s & 1) ^ 1) ? MESH_BUF : 0));
            __syncthreads();
        }
    }
    if (!live) return;
    const double ux = scale[2 * IT.traj], uz = scale[2 * IT.traj + 1];
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

extern "C" int srwd_launch_sr_mesh(const srwd_item* dItems, const int2* dTiles, int ntU, int nTiles, const srwd_trj_info* dInfo,
                                   const srwd_mrec* dRec, long long ldM, const double* dScale, int nSplit,
                                   long long nPointsPad, double* dPart, hipStream_t st)
{
    if (nTiles <= 0) return 0;
    hipLaunchKernelGGL(k_sr_mesh, dim3(nTiles, nSplit), dim3(256), 0, st, dItems, dTiles, ntU, dInfo, dRec, ldM, dScale, nSplit,
                       nPointsPad, dPart);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

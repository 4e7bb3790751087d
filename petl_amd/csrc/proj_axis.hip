// Separable projectors for psi = 0 or 90 degrees and any voxel size (see proj_axis.h).
//
// axis_fwd_kernel: a workgroup of 8 waves takes 4 u1 rows of a view row v1 and up to 64 (view, 64-bin) items, 8 per wave.
//   Per block of slices the volume is interpolated along z onto the 4 rows into LDS, one 16-byte cell per (slice,
//   in-plane index); each lane then forms its bin's overlaps once and applies them to the 4 rows (one 16-byte LDS read and
//   four multiply-adds per cell).  Bound by the overlaps' vector work and those reads.
// axis_back_u0_kernel: a wave takes 64 columns (slice, in-plane) and 8 u1 rows of one v1; per view the lane's bins and
//   overlaps are formed once and applied to the 8 rows.  Bound by its loads of planogram rows from L1.
// axis_back_z_kernel: a workgroup takes 64 columns and 2 heights, each wave a quarter of the v1 rows, summed in wave order.
//
// Pair of a 32^3 volume at 3 mm with two (47, 75, 48, 122) planograms of 2 mm crystals, per planogram: forward 146 us
// (the per-bin general kernel 1.32 ms: nothing shared between rows), back 115 + 23 us (19.8 ms: 8192 threads in all,
// every one walking all views).  A 60-crystal pair on 4 mm voxels in matched mode 37.6 -> 0.96 ms, a 40-crystal pair on
// 1.6 mm voxels 15.2 -> 0.53 ms.
#include <algorithm>
#include <cmath>
#include "proj_axis.h"
#include "proj_kernels.h"
#include "proj_general_dev.h"

namespace petl {

namespace {

constexpr int AX_R = 4;      // u1 rows per forward workgroup
constexpr int AX_NI = 8;     // (view, 64-bin) items per forward wave
constexpr int AX_WAVES = 8;  // waves per forward workgroup
constexpr int AX_SB = 8;     // slices per LDS block at most
constexpr int AX_RB = 8;     // u1 rows per wave of the u0 gather
constexpr int AX_ZC = 2;     // heights per workgroup of the z gather
constexpr size_t AX_LDS = 60 * 1024;
constexpr size_t AX_WS = size_t(1) << 30;

struct AxisArgs {
    GenArgs G;
    int xs, Ns, Na;  // slices along x (and in-plane along y) or the other way round
    float Au, hb;    // crossing per bin and half width in voxels, the same for all views
    int sb;          // slices per LDS block
    int nv1;         // v1 rows of this launch: G.v1_first + (G.v1_chunk + k) * G.v1_stride
};

// cells of a bin (forward) and bins of a voxel (back, in either mode) at most
inline int cells_of(float hb) { return int(std::ceil(2.0 * double(hb) - 1e-6)) + 1; }

// ---------------------------------------------------------------------------------------------------------
// forward
// ---------------------------------------------------------------------------------------------------------
template <int NA>
__global__ void __launch_bounds__(64 * AX_WAVES) axis_fwd_kernel(float* __restrict__ g, const float* __restrict__ vol,
                                                                 AxisArgs A, int epilogue, const float* __restrict__ y,
                                                                 const float* __restrict__ resp,
                                                                 const float* __restrict__ wts)
{
    extern __shared__ __align__(16) float4 s_h[];  // [slice of the block][NA zeros, Na cells, NA zeros]
    const PlanGeom& P = A.G.P;
    const VolGeom& V = A.G.V;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nc = (P.Nu0 + 63) >> 6, nitems = P.Nv0 * nc;
    const int item0 = (int(blockIdx.x) * AX_WAVES + wave) * AX_NI;
    const int iu1_0 = blockIdx.y * AX_R;
    const int iv1 = A.G.v1_first + (A.G.v1_chunk + int(blockIdx.z)) * A.G.v1_stride;
    const float v1 = coord(iv1, P.Tv1, P.v1_0);
    const int Ns = A.Ns, Na = A.Na, Nz = V.Nz, pitch = Na + 2 * NA;
    const GenView wm = A.G.views[int64_t(iv1) * P.Nv0 + P.Nv0 / 2];  // z crossings: the same for all views
    const float hz = A.G.hz, Bz = A.G.Bz;
    bool live[AX_R];
    bool any = false;
#pragma unroll
    for (int r = 0; r < AX_R; r++) {
        live[r] = iu1_0 + r < P.Nu1 && !mask_u1(P, coord(iu1_0 + r, P.Tu1, P.u1_0), v1);
        any = any || live[r];
    }
    float acc[AX_NI][AX_R];
#pragma unroll
    for (int j = 0; j < AX_NI; j++)
#pragma unroll
        for (int r = 0; r < AX_R; r++)
            acc[j][r] = 0.0f;
    if (any) {
        for (int i = tid; i < A.sb * 2 * NA; i += 64 * AX_WAVES) {
            const int r = i / (2 * NA), k = i - r * 2 * NA;
            s_h[r * pitch + (k < NA ? k : Na + k)] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
        const int64_t sk = int64_t(Ns) * Na;
        for (int sb = 0; sb < Ns; sb += A.sb) {
            const int ns = min(A.sb, Ns - sb);
            // heights that the rows cross in this block's slices (with a voxel of margin): none inside, nothing to add
            const float za = fmaf(wm.Bs, float(sb), wm.Z0), ze = fmaf(wm.Bs, float(sb + ns - 1), wm.Z0);
            const float zl = fminf(za, ze) + Bz * float(iu1_0), zh = fmaxf(za, ze) + Bz * float(iu1_0 + AX_R - 1);
            if (zh + hz + 1.5f < 0.0f || zl - hz - 1.5f > float(Nz - 1))
                continue;
            __syncthreads();
            for (int idx = tid; idx < ns * Na; idx += 64 * AX_WAVES) {
                const int sl = idx / Na, a = idx - sl * Na, s = sb + sl;
                const float* vs = vol + int64_t(s) * Na + a;
                float h[AX_R];
#pragma unroll
                for (int r = 0; r < AX_R; r++) {
                    h[r] = 0.0f;
                    const float c = cross_z(Bz, fmaf(wm.Bs, float(s), wm.Z0), iu1_0 + r);
                    const int klo = max(0, int(floorf(c - hz + 0.5f))), khi = min(Nz - 1, int(ceilf(c + hz - 0.5f)));
                    if (live[r])
                        for (int k = klo; k <= khi; k++)
                            h[r] += vs[int64_t(k) * sk] * fmaxf(0.0f, overlap(c, hz, float(k)));
                }
                s_h[sl * pitch + NA + a] = make_float4(h[0], h[1], h[2], h[3]);
            }
            __syncthreads();
#pragma unroll
            for (int j = 0; j < AX_NI; j++) {
                const int item = item0 + j;
                if (item < nitems) {
                    const int v = item / nc, c = item - v * nc;
                    const float* xr = A.G.xi0 + int64_t(v) * A.G.Nsmax + sb;
                    const float pf = float(c * 64 + lane);
                    for (int sl = 0; sl < ns; sl++) {
                        const float xi = fmaf(A.Au, pf, xr[sl]);
                        const int i0 = int(floorf(xi + (0.5f - A.hb)));
                        const float4* cell = s_h + sl * pitch + NA + min(max(i0, -NA), Na);
#pragma unroll
                        for (int k = 0; k < NA; k++) {
                            const float w = fmaxf(0.0f, overlap(xi, A.hb, float(i0 + k)));
                            const float4 h = cell[k];
                            acc[j][0] += w * h.x;
                            acc[j][1] += w * h.y;
                            acc[j][2] += w * h.z;
                            acc[j][3] += w * h.w;
                        }
                    }
                }
            }
        }
    }
    static_assert(AX_NI * AX_R <= 32, "a bit per bin of a lane");
    unsigned again = 0;
#pragma unroll
    for (int j = 0; j < AX_NI; j++) {
        const int item = item0 + j;
        const int v = item / nc, iu0 = (item - v * nc) * 64 + lane;
        if (item < nitems && iu0 < P.Nu0) {
            const bool in = !mask_u0(P, coord(iu0, P.Tu0, P.u0_0), coord(v, P.Tv0, P.v0_0));
            const float scale = A.G.views[int64_t(iv1) * P.Nv0 + v].scale;
#pragma unroll
            for (int r = 0; r < AX_R; r++)
                if (iu1_0 + r < P.Nu1) {
                    const int64_t gi = ((int64_t(iv1) * P.Nv0 + v) * P.Nu1 + iu1_0 + r) * P.Nu0 + iu0;
                    if (in && live[r] && !__builtin_isfinite(acc[j][r]))
                        again |= 1u << (j * AX_R + r);
                    else
                        g[gi] = gen_epilogue(in && live[r] ? acc[j][r] * scale : 0.0f, gi, epilogue, y, resp, wts);
                }
        }
    }
    // A cell beside the footprint has the weight zero, which an infinity or a NaN would turn into a NaN: a bin that came out
    // as one is summed again, over the cells that it meets.
    const int64_t sk = int64_t(Ns) * Na;
    for (; again; again &= again - 1) {
        const int b = __ffs(again) - 1, item = item0 + b / AX_R, v = item / nc, iu0 = (item - v * nc) * 64 + lane;
        const int iu1 = iu1_0 + b % AX_R;
        float sum = 0.0f;
        for (int s = 0; s < Ns; s++) {
            const float xi = fmaf(A.Au, float(iu0), A.G.xi0[int64_t(v) * A.G.Nsmax + s]);
            const float c = cross_z(Bz, fmaf(wm.Bs, float(s), wm.Z0), iu1);
            const int i0 = int(floorf(xi + (0.5f - A.hb)));
            const int klo = max(0, int(floorf(c - hz + 0.5f))), khi = min(Nz - 1, int(ceilf(c + hz - 0.5f)));
            for (int a = max(i0, 0); a < min(i0 + NA, Na); a++) {
                const float w = overlap(xi, A.hb, float(a));
                float h = 0.0f;
                for (int k = klo; k <= khi && w > 0.0f; k++) {
                    const float wz = overlap(c, hz, float(k));
                    if (wz > 0.0f)
                        h += vol[int64_t(k) * sk + int64_t(s) * Na + a] * wz;
                }
                if (w > 0.0f)
                    sum += w * h;
            }
        }
        const int64_t gi = ((int64_t(iv1) * P.Nv0 + v) * P.Nu1 + iu1) * P.Nu0 + iu0;
        g[gi] = gen_epilogue(sum * A.G.views[int64_t(iv1) * P.Nv0 + v].scale, gi, epilogue, y, resp, wts);
    }
}

// ---------------------------------------------------------------------------------------------------------
// back projection, stage 1: the bins of every v0 into columns, h2[v1 of the launch][u1][slice][in-plane]
// ---------------------------------------------------------------------------------------------------------
template <int NP, bool MATCHED>
__global__ void __launch_bounds__(256) axis_back_u0_kernel(const float* __restrict__ g, float* __restrict__ h2, AxisArgs A)
{
    const PlanGeom& P = A.G.P;
    const VolGeom& V = A.G.V;
    const int Na = A.Na, ncol = A.Ns * Na;
    const int col = blockIdx.x * 256 + threadIdx.x, colc = min(col, ncol - 1);
    const int s = colc / Na, a = colc - s * Na;
    const int iu1_0 = blockIdx.y * AX_RB;
    const int iv1 = A.G.v1_first + (A.G.v1_chunk + int(blockIdx.z)) * A.G.v1_stride;
    const float x = coord(A.xs ? s : a, V.Tx, V.x0), yv = coord(A.xs ? a : s, V.Ty, V.y0);
    const float fa = float(a);
    const int rmax = min(AX_RB, P.Nu1 - iu1_0) - 1;
    const unsigned rowb = unsigned(P.Nu0);
    float acc[AX_RB];
#pragma unroll
    for (int r = 0; r < AX_RB; r++)
        acc[r] = 0.0f;
    const GenView* wr = A.G.views + int64_t(iv1) * P.Nv0;
    // the column's bins in view iv0, p0 ... p0 + NP - 1, and their weights (zero outside its footprint)
    auto weights = [&](int iv0, float(&w)[NP]) {
        int p0;
        if (MATCHED) {
            // bins whose footprint meets cell a: crossings within hb + 1/2 of it (one bin of margin below)
            const float xs0 = A.G.xi0[int64_t(iv0) * A.G.Nsmax + s], v0 = coord(iv0, P.Tv0, P.v0_0);
            p0 = min(max(int(floorf((fa - A.hb - 0.5f - xs0) / A.Au)), 0), P.Nu0 - NP);
#pragma unroll
            for (int k = 0; k < NP; k++) {
                const float o = overlap(fmaf(A.Au, float(p0 + k), xs0), A.hb, fa);
                w[k] = (o > 0.0f && !mask_u0(P, coord(p0 + k, P.Tu0, P.u0_0), v0)) ? o * wr[iv0].scale : 0.0f;
            }
        } else {
            const float4 pc = A.G.pcoef[iv0];
            const float c0 = fmaf(x, pc.x, fmaf(yv, pc.y, pc.z)), A0 = c0 - pc.w, B0 = c0 + pc.w;
            p0 = min(max(int(ceilf(A0 - 0.5f)), 0), P.Nu0 - NP);
#pragma unroll
            for (int k = 0; k < NP; k++)
                w[k] = fmaxf(0.0f, fminf(float(p0 + k) + 0.5f, B0) - fmaxf(float(p0 + k) - 0.5f, A0)) * wr[iv0].lpetl;
        }
        return p0;
    };
    const float* g1 = g + (int64_t(iv1) * P.Nv0 * P.Nu1 + iu1_0) * P.Nu0;
    for (int iv0 = 0; iv0 < P.Nv0; iv0++) {
        float w[NP];
        const int p0 = weights(iv0, w);
        const float* gv = g1 + int64_t(iv0) * P.Nu1 * P.Nu0;
#pragma unroll
        for (int r = 0; r < AX_RB; r++) {
            const float* q = gv + unsigned(min(r, rmax)) * rowb + unsigned(p0);
#pragma unroll
            for (int k = 0; k < NP; k++)
                acc[r] += w[k] * q[k];
        }
    }
    // A bin beside the footprint has the weight zero, which an infinity or a NaN would turn into a NaN: columns that come out
    // as one are summed again, over the bins that they meet.
    bool void_row = false;
#pragma unroll
    for (int r = 0; r < AX_RB; r++)
        void_row = void_row || !__builtin_isfinite(acc[r]);
    if (void_row) {
#pragma unroll
        for (int r = 0; r < AX_RB; r++)
            acc[r] = 0.0f;
#pragma unroll 1
        for (int iv0 = 0; iv0 < P.Nv0; iv0++) {
            float w[NP];
            const int p0 = weights(iv0, w);
            const float* gv = g1 + int64_t(iv0) * P.Nu1 * P.Nu0;
#pragma unroll
            for (int r = 0; r < AX_RB; r++) {
                const float* q = gv + unsigned(min(r, rmax)) * rowb + unsigned(p0);
#pragma unroll
                for (int k = 0; k < NP; k++) {
                    const float x1 = w[k] > 0.0f ? q[k] : 0.0f;
                    acc[r] += w[k] * x1;
                }
            }
        }
    }
    if (col < ncol) {
        float* o = h2 + (int64_t(blockIdx.z) * P.Nu1 + iu1_0) * ncol + col;
#pragma unroll
        for (int r = 0; r < AX_RB; r++)
            if (r <= rmax)
                o[int64_t(r) * ncol] = acc[r];
    }
}

// ---------------------------------------------------------------------------------------------------------
// back projection, stage 2: the u1 rows of every v1 into the voxels, f += sum
// ---------------------------------------------------------------------------------------------------------
template <bool MATCHED>
__global__ void __launch_bounds__(256) axis_back_z_kernel(const float* __restrict__ h2, float* __restrict__ f, AxisArgs A)
{
    __shared__ float s_sum[3][AX_ZC][64];
    const PlanGeom& P = A.G.P;
    const VolGeom& V = A.G.V;
    const int Na = A.Na, ncol = A.Ns * Na;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = blockIdx.x * 64 + lane, colc = min(col, ncol - 1);
    const int s = colc / Na, a = colc - s * Na;
    const int ix = A.xs ? s : a, iy = A.xs ? a : s;
    const int z0 = blockIdx.y * AX_ZC;
    float tcol;
    {
#pragma clang fp contract(off)
        // the voxel centre's signed distance along the panel normal direction (src/projectors.cu:284)
        tcol = coord(iy, V.Ty, V.y0) * P.cos_psi - coord(ix, V.Tx, V.x0) * P.sin_psi;
    }
    const float hz1 = 0.5f * V.Tz / P.Tu1, hz = A.G.hz, Bz = A.G.Bz;
    float acc[AX_ZC];
#pragma unroll
    for (int j = 0; j < AX_ZC; j++)
        acc[j] = 0.0f;
    for (int k1 = wave; k1 < A.nv1; k1 += 4) {
        const int iv1 = A.G.v1_first + (A.G.v1_chunk + k1) * A.G.v1_stride;
        const float v1 = coord(iv1, P.Tv1, P.v1_0);
        const float* hv = h2 + int64_t(k1) * P.Nu1 * ncol + colc;
        const GenView wm = A.G.views[int64_t(iv1) * P.Nv0 + P.Nv0 / 2];
        const float zb = fmaf(wm.Bs, float(s), wm.Z0);
#pragma unroll
        for (int j = 0; j < AX_ZC; j++) {
            const int iz = z0 + j;
            if (MATCHED) {
                const float fz = float(iz);
                const int r0 = max(0, int(floorf((fz - hz - 0.5f - zb) / Bz)) - 1);
                const int r1 = (iz < V.Nz) ? min(P.Nu1 - 1, int(ceilf((fz + hz + 0.5f - zb) / Bz)) + 1) : -1;
                for (int r = r0; r <= r1; r++) {
                    const float wz = overlap(cross_z(Bz, zb, r), hz, fz);
                    if (wz > 0.0f && !mask_u1(P, coord(r, P.Tu1, P.u1_0), v1))
                        acc[j] += wz * hv[int64_t(r) * ncol];
                }
            } else {
                float u1;
                bool live;
                {
#pragma clang fp contract(off)
                    u1 = coord(iz, V.Tz, V.z0) + v1 * tcol;
                    live = (iz < V.Nz) && !(fabsf(u1) - 0.5f * P.Tu1 > P.H - P.R * fabsf(v1));
                }
                const float mid = (u1 - P.u1_0) / P.Tu1, A1 = mid - hz1, B1 = mid + hz1;
                const int r0 = max(0, int(ceilf(A1 - 0.5f)));
                const int r1 = live ? min(P.Nu1 - 1, int(floorf(B1 + 0.5f))) : -1;
                for (int r = r0; r <= r1; r++) {
                    const float w1 = fmaxf(0.0f, fminf(float(r) + 0.5f, B1) - fmaxf(float(r) - 0.5f, A1));
                    if (w1 > 0.0f)
                        acc[j] += w1 * hv[int64_t(r) * ncol];
                }
            }
        }
    }
    if (wave > 0)
#pragma unroll
        for (int j = 0; j < AX_ZC; j++)
            s_sum[wave - 1][j][lane] = acc[j];
    __syncthreads();
    if (wave == 0 && col < ncol)
#pragma unroll
        for (int j = 0; j < AX_ZC; j++)
            if (z0 + j < V.Nz) {
                const float t = ((acc[j] + s_sum[0][j][lane]) + s_sum[1][j][lane]) + s_sum[2][j][lane];
                f[(int64_t(z0 + j) * V.Ny + iy) * V.Nx + ix] += MATCHED ? t : V.Tx * t;
            }
}

AxisArgs axis_args(const GenPlan& gp, int v1_first, int v1_stride)
{
    AxisArgs A;
    A.G = gen_args(gp, v1_first, v1_stride);
    A.xs = gp.axis_xs;
    A.Ns = gp.axis_xs ? gp.V.Nx : gp.V.Ny;
    A.Na = gp.axis_xs ? gp.V.Ny : gp.V.Nx;
    A.Au = gp.axis_Au;
    A.hb = gp.axis_hb;
    A.sb = 0;
    A.nv1 = (gp.P.Nv1 - v1_first + v1_stride - 1) / v1_stride;
    return A;
}

// bins per voxel in each mode (matched: one of margin for the rounding of the first)
inline int back_bins(const GenPlan& gp, int mode)
{
    const double r = 2.0 * double(gp.axis_hb);
    return mode == BACK_MATCHED ? int(std::ceil((1.0 + r) / r - 1e-6)) + 1 : cells_of(gp.axis_h0);
}

int64_t rows_per_pass(const PlanGeom& P, const VolGeom& V)
{
    const size_t one = size_t(P.Nu1) * V.Nx * V.Ny * sizeof(float);
    return std::max<int64_t>(1, std::min<int64_t>(P.Nv1, int64_t(AX_WS / one)));
}

}  // namespace

bool axis_eligible(const GenPlan& gp)
{
    if (gp.axis_xs < 0)
        return false;
    const int Na = gp.axis_xs ? gp.V.Ny : gp.V.Nx, na = cells_of(gp.axis_hb);
    const int np = std::max(back_bins(gp, BACK_PETL), back_bins(gp, BACK_MATCHED));
    return gp.axis_hb > 0.0f && na <= 4 && np <= 5 && gp.P.Nu0 >= 5 &&
           size_t(Na + 2 * na) * sizeof(float4) <= AX_LDS && gp.P.Nv0 > 0;
}

void axis_forward(const GenPlan& gp, float* g, const float* vol, int epilogue, const float* y, const float* resp,
                  const float* wts, hipStream_t s, int v1_first, int v1_stride)
{
    AxisArgs A = axis_args(gp, v1_first, v1_stride);
    const int na = std::max(2, cells_of(gp.axis_hb)), pitch = A.Na + 2 * na;
    A.sb = std::max(1, std::min({AX_SB, A.Ns, int(AX_LDS / (size_t(pitch) * sizeof(float4)))}));
    const size_t lds = size_t(A.sb) * pitch * sizeof(float4);
    const int items = gp.P.Nv0 * ((gp.P.Nu0 + 63) / 64), per = AX_NI * AX_WAVES;
    auto fn = na == 2 ? axis_fwd_kernel<2> : na == 3 ? axis_fwd_kernel<3> : axis_fwd_kernel<4>;
    const int nv1 = A.nv1;
    for (int c = 0; c < nv1; c += 65535) {
        A.G.v1_chunk = c;
        hipLaunchKernelGGL(fn, dim3((items + per - 1) / per, (gp.P.Nu1 + AX_R - 1) / AX_R, std::min(65535, nv1 - c)),
                           dim3(64 * AX_WAVES), lds, s, g, vol, A, epilogue, y, resp, wts);
        PETL_LAUNCH_CHECK();
    }
}

size_t axis_back_workspace_bytes(const PlanGeom& P, const VolGeom& V)
{
    return size_t(rows_per_pass(P, V)) * P.Nu1 * V.Nx * V.Ny * sizeof(float);
}

void axis_back(const GenPlan& gp, const float* g, float* f, int mode, hipStream_t s, int v1_first, int v1_stride,
               float* workspace)
{
    AxisArgs A = axis_args(gp, v1_first, v1_stride);
    const int nv1 = A.nv1, ncol = A.Ns * A.Na, np = back_bins(gp, mode);
    const int64_t per = std::min<int64_t>(rows_per_pass(gp.P, gp.V), 65535);
    using u0_fn = void (*)(const float*, float*, AxisArgs);
    const u0_fn petl[] = {axis_back_u0_kernel<2, false>, axis_back_u0_kernel<3, false>, axis_back_u0_kernel<4, false>,
                          axis_back_u0_kernel<5, false>};
    const u0_fn matched[] = {axis_back_u0_kernel<3, true>, axis_back_u0_kernel<3, true>, axis_back_u0_kernel<4, true>,
                             axis_back_u0_kernel<5, true>};
    const u0_fn u0 = (mode == BACK_MATCHED ? matched : petl)[std::max(2, np) - 2];
    for (int64_t c = 0; c < nv1; c += per) {
        A.G.v1_chunk = int(c);
        A.nv1 = int(std::min<int64_t>(per, nv1 - c));
        hipLaunchKernelGGL(u0, dim3((ncol + 255) / 256, (gp.P.Nu1 + AX_RB - 1) / AX_RB, A.nv1), dim3(256), 0, s, g,
                           workspace, A);
        PETL_LAUNCH_CHECK();
        const dim3 zgrid((ncol + 63) / 64, (gp.V.Nz + AX_ZC - 1) / AX_ZC);
        if (mode == BACK_MATCHED)
            hipLaunchKernelGGL(axis_back_z_kernel<true>, zgrid, dim3(256), 0, s, workspace, f, A);
        else
            hipLaunchKernelGGL(axis_back_z_kernel<false>, zgrid, dim3(256), 0, s, workspace, f, A);
        PETL_LAUNCH_CHECK();
    }
}

}  // namespace petl

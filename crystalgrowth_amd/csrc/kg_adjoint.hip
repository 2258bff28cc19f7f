// kg_adjoint.hip -- reverse-mode (adjoint) of the Kobayashi step.
//
// Loss L = sum over cells of (phi_N - target)^2 after N steps, accumulated in
// FP64.  One reverse step maps the adjoint of the step's outputs
// (lphi', lT', ltheta') to the adjoint of its inputs (lphi, lT, ltheta_old)
// and adds the step's contribution to dL/d(parameter).  Derivation, with
// s = t1 + t2 + e^2 lap + t3 + r the bracket of src/Kobayashi.cpp:211-214,
// phi' = phi + s dt/tau, T' = T + lapT dt + K (phi' - phi):
//   ls        = (lphi' + K lT') dt/tau                          (adjoint of s)
//   l(e^2)(c) = sum over readers k of s(k):  +-ls(k) g(k)/dx (gEx, gEy) + ls(c) lap(c)
//   lA(c)     = ls(S-reader) / dy - ls(N-reader) / dy   (t1),   lB similarly (t2)
//   ltheta    = l(e^2) 2 e e' + (lA gx + lB gy)(e'^2 + e e'') + ltheta'
//   theta = atan branch: lgx += ltheta (-gy/|g|^2), lgy += ltheta gx/|g|^2
//   theta not rewritten (src/Kobayashi.cpp:154-167): ltheta_old = ltheta
//   lphi, lT  = gathers of lgx, lgy, ls e^2 (9-point) and lT' dt (9-point)
//               through the inverse neighbour maps, plus the local terms.
// "Readers" enumerate the inverse of the boundary map: periodic has one
// reader per direction; zero-flux boundary cells are also read by themselves.
// Every kernel is a gather (no atomics), so results are deterministic.
//
// Checkpoint-and-recompute: the forward run stores (phi, T, theta) every
// `every` steps; the reverse pass recomputes each segment's states with the
// same step kernels (bitwise identical) and walks them backwards.  The last
// segment is stepped straight into the segment's buffers, so it is not
// recomputed; small grids and batches store a segment's states from launches of
// three steps.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <functional>
#include <string>
#include <vector>

#include "kg_host.h"
#include "kg_math.h"
#include "kg_philox.h"

namespace kg {

namespace {

enum { P_TAU, P_EPS_BAR, P_K, P_DELTA, P_THETA0, P_ALPHA, P_GAMMA, P_TEQ, P_NOISE, NPAR };

template <typename R>
struct AdjIO {
    const R *phi, *T, *theta_old;   // the step's input state
    const R *lphi1, *lT1, *lth1;    // adjoint of the step's outputs
    R *lphi0, *lT0, *lth0;          // adjoint of the step's inputs
    // one word per tile and adjoint buffer: 1 when all three adjoints are 0
    // on the tile (0: not known to be)
    const uint32_t *zero1;          // of lphi1, lT1, lth1
    uint32_t *zero0;                // of lphi0, lT0, lth0 (before and after the step)
};

template <int BC>
__device__ __forceinline__ int map_index(int x, int n)
{
    if (BC == 1)
        return x < 0 ? 0 : (x >= n ? n - 1 : x);
    while (x < 0)
        x += n;
    while (x >= n)
        x -= n;
    return x;
}

template <typename R> __device__ __forceinline__ R pi_of();
template <> __device__ __forceinline__ float pi_of<float>() { return 3.14159274f; }
template <> __device__ __forceinline__ double pi_of<double>() { return 3.14159265358979323846; }

// theta update of src/Kobayashi.cpp:154-167 with the branch class:
// 0 = theta kept, 1 = offset + atan(gy/gx), 2 = +-pi/2.
template <typename R>
__device__ __forceinline__ int theta_class(R gx, R gy, R &th)
{
    const R E = (R)1.1920928955078125e-7;
    const R PI = pi_of<R>();
    const bool yneg = gy < -E, ypos = gy > E, xneg = gx < -E;
    if (xneg || (gx > E && (yneg || ypos))) {
        const R t = kg_atan_ratio(gy, gx);
        th = xneg ? PI + t : (yneg ? (R)2.0 * PI + t : t);
        return 1;
    }
    if (gx <= E && gx >= -E && (yneg || ypos)) {
        th = yneg ? (R)-0.5 * PI : (R)0.5 * PI;
        return 2;
    }
    return 0;
}

// (2 (E + W + N + S) + NE + SW + NW + SE - 12 C) around p[0], rows w apart
template <typename R>
__device__ __forceinline__ R lap9(const R *p, int w)
{
    return (R)2.0 * (p[1] + p[-1] + p[w] + p[-w]) + p[w + 1] + p[-w - 1] + p[w - 1] + p[-w + 1] -
           (R)12.0 * p[0];
}

// Sum of v over the 16 lanes of a DPP row, in every lane (quad swaps, then
// row rotations by 4 and 8).
template <int CTRL>
__device__ __forceinline__ double dpp(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, false);
    return __longlong_as_double((long long)hi << 32 | (unsigned)lo);
}
__device__ __forceinline__ double row_sum(double v)
{
    v += dpp<0xB1>(v);   // quad_perm [1,0,3,2]
    v += dpp<0x4E>(v);   // quad_perm [2,3,0,1]
    v += dpp<0x124>(v);  // row_ror:4
    v += dpp<0x128>(v);  // row_ror:8
    return v;
}

// One reverse step of a 32 x 8 tile, all of it in one launch: phi is staged
// with a halo of 3 cells, the rest with 2; the forward pass-1 quantities of
// the 2-cell halo, the reverse of pass 2 on the tile, of pass 1 on the 1-cell
// halo and the gather of the input adjoints follow in LDS.  Per cell a step
// reads phi, T, theta and three adjoints and writes three (36 B in FP32);
// four kernels through 17 temporary fields moved some 200 B.  us per step:
// 512^2 FP32 30 -> 7.7, 24 members of 128^2 .. 512^2 (2.6 M cells) 184 -> 27.
// Bound by a tile's chain of loads and four barriers (0.19 of the VALU's issue
// slots at 512^2, 0.53 on the members) and by VALU work (1.7 pass-1 cells per
// output cell).  Tiles and threads measured on whole
// adjoints, us (512^2 FP32 / FP64, the 24 members FP32 / FP64, 190 x 133
// FP64): 32 x 8 on 256 threads 3725 / 5165 / 8380 / 17045 / 1537, on 512
// 3647 / 5584 / 9353 / 19442 / 1431; 32 x 16 on 256 3960 / 5290 / 7847 /
// 16503 / 1650, on 768 3704 / 5666 / 8993 / 21441 / 1517; 32 x 32 on 512
// 3846 / 5264 / 8494 / 20160 / 1766.  One shape for all, so that a member's
// sums group alike in a batch and alone.  Asking for 6 or 8 waves per SIMD
// (it takes 5) was slower: 3666 -> 4054 and 4074.
constexpr int AX = 32, AY = 8, ANT = 256;      // tile, threads
constexpr int PW = AX + 6, PN = PW * (AY + 6);  // staged phi
constexpr int QW = AX + 4, QN = QW * (AY + 4);  // everything else in LDS
constexpr int ON = AX * AY;
constexpr int TP = (PN + ANT - 1) / ANT, TQ = (QN + ANT - 1) / ANT;  // trips
static_assert(ON == ANT && ANT % 64 == 0 && ANT >= 16 * NPAR, "one output cell per thread");

template <typename R>
struct AdjSmem {
    R P[PN];
    R E2[QN];  // eps^2, then ls eps^2
    R F[QN];   // eps eps'
    R GX[QN];  // gx, then its adjoint
    R GY[QN];  // gy, then its adjoint
    R LS[QN];  // adjoint of the bracket s
    R LT[QN];  // lT1
    R X[ON];   // chi
    double red[NPAR][ANT / 16];
    int W[ANT / 64];
};

// Zero-flux boundaries: a ghost cell stands for the cell it clamps to.  The
// 9-point gathers are their own transpose under the clamp, so ghosts of ls
// eps^2 and lT1 hold that cell's value; a central difference under the clamp
// transposes to itself with the ghost's sign turned (the cell reads itself
// once with each sign), so ghosts of ls and of the gradients' adjoints hold
// its negative.
template <typename R, int BC, bool ASK>
__device__ __forceinline__ void adj_tile(const AdjMember<R> &m, const AdjIO<R> &io, int x0, int y0,
                                         uint32_t step, double *__restrict__ acc, int nslots,
                                         int slot, bool first, AdjSmem<R> &sm)
{
    const StepArgs<R> &a = m.a;
    const int nx = a.nx, ny = a.ny, tid = threadIdx.x;
    const bool interior = x0 >= 3 && y0 >= 3 && x0 + AX + 3 <= nx && y0 + AY + 3 <= ny;
    auto cell = [&](int ux, int uy) -> size_t {
        if (!interior) {
            ux = map_index<BC>(ux, nx);
            uy = map_index<BC>(uy, ny);
        }
        return m.off + (size_t)uy * nx + ux;
    };
    // this thread's output cell
    const int rw = tid / AX, cw = tid - rw * AX, i = x0 + cw, j = y0 + rw;
    const bool own = i < nx && j < ny;
    const size_t oo = m.off + (size_t)j * nx + i;
    // this block's running sums, loaded with everything else
    const bool adder = tid < 16 * NPAR && (tid & 15) == 0;
    double *const sum = acc + (size_t)(tid >> 4) * nslots + slot;
    const double before = adder && !first ? *sum : 0.0;

    // The adjoint of a step reaches 2 cells further than that of its output,
    // so a tile whose 3 x 3 neighbourhood is all zero stays zero and has
    // nothing to add.  ASK: lanes 0..8 of a wave ask for the neighbourhood
    // before anything is loaded, lane 9 for what the output buffers already
    // hold.  Periodic grids whose last tile is one cell wide reach past it.
    const bool words = ASK && (BC == 1 || (nx % AX != 1 && ny % AY != 1));
    bool zeros = false;  // the output buffers already hold zeros here
    if (words) {
        const int tx = x0 / AX, ty = y0 / AY, lane = tid & 63;
        const int tiles_x = (nx + AX - 1) / AX, tiles_y = (ny + AY - 1) / AY;
        const int ln = lane < 9 ? lane : 4;
        const int nb = slot + (map_index<BC>(ty + ln / 3 - 1, tiles_y) - ty) * tiles_x +
                       map_index<BC>(tx + ln % 3 - 1, tiles_x) - tx;
        const uint32_t word = lane < 9 ? io.zero1[nb] : io.zero0[slot];
        zeros = __builtin_amdgcn_readlane((int)word, 9) != 0;
        if ((__ballot(lane < 9 && word != 0) & 0x1ffull) == 0x1ffull) {
            if (adder && first)
                *sum = 0.0;
            if (!zeros) {
                if (own) {
                    io.lphi0[oo] = (R)0;
                    io.lT0[oo] = (R)0;
                    io.lth0[oo] = (R)0;
                }
                __syncthreads();  // every wave has read the word before it changes
                if (tid == 0)
                    io.zero0[slot] = 1u;
            }
            return;
        }
    }
    R vp[TP], th[TQ], lp[TQ], lT[TQ], lth[TQ], Tc = (R)0, lp1 = (R)0;
#pragma unroll
    for (int t = 0; t < TP; ++t) {
        const int k = tid + t * ANT, r = k / PW, c = k - r * PW;
        vp[t] = k < PN ? io.phi[cell(x0 - 3 + c, y0 - 3 + r)] : (R)0;
    }
    bool nonzero = false;
#pragma unroll
    for (int t = 0; t < TQ; ++t) {
        const int k = tid + t * ANT, r = k / QW, c = k - r * QW;
        th[t] = lp[t] = lT[t] = lth[t] = (R)0;
        if (k < QN) {
            const size_t o = cell(x0 - 2 + c, y0 - 2 + r);
            th[t] = io.theta_old[o];
            lp[t] = io.lphi1[o];
            lT[t] = io.lT1[o];
            lth[t] = io.lth1[o];
        }
    }
    if (own) {
        Tc = io.T[oo];
        lp1 = io.lphi1[oo];
    }
#pragma unroll
    for (int t = 0; t < TP; ++t)
        if (tid + t * ANT < PN)
            sm.P[tid + t * ANT] = vp[t];
#pragma unroll
    for (int t = 0; t < TQ; ++t)
        nonzero |= lp[t] != (R)0 || lT[t] != (R)0 || lth[t] != (R)0;
    {
        const bool w = __ballot(nonzero) != 0;
        if ((tid & 63) == 0)
            sm.W[tid >> 6] = w ? 1 : 0;
    }
    __syncthreads();
    int any = 0;
#pragma unroll
    for (int w = 0; w < ANT / 64; ++w)
        any |= sm.W[w];
    if (!any) {  // every adjoint that reaches the tile is zero: so are its inputs'
        if (own && !zeros) {
            io.lphi0[oo] = (R)0;
            io.lT0[oo] = (R)0;
            io.lth0[oo] = (R)0;
        }
        if (adder && first)
            *sum = 0.0;
        if (words && tid == 0)
            io.zero0[slot] = 1u;  // (after the barrier: every wave has read it)
        return;
    }
    if (words && tid == 0)
        io.zero0[slot] = 0u;

    // ---- forward pass 1 on the 2-cell halo -------------------------------
    // own cell's values, kept for the reverse of pass 1
    R gx[TQ], gy[TQ], eps[TQ], epsd[TQ], cs[TQ], sn[TQ];
    int code[TQ], ctr[TQ];  // branch class; LDS index of the cell (a ghost's: of its cell)
    bool ghost[TQ];
#pragma unroll
    for (int t = 0; t < TQ; ++t) {
        const int k = tid + t * ANT;
        if (k >= QN)
            continue;
        const int r = k / QW, c = k - r * QW;
        int lr = r, lc = c;
        ghost[t] = false;
        if (BC == 1 && !interior) {
            const int ux = x0 - 2 + c, uy = y0 - 2 + r;
            lr += map_index<1>(uy, ny) - uy;
            lc += map_index<1>(ux, nx) - ux;
            ghost[t] = lr != r || lc != c;
        }
        ctr[t] = lr * QW + lc;
        const R *p = &sm.P[(lr + 1) * PW + lc + 1];
        gx[t] = (p[1] - p[-1]) * a.inv_dx;
        gy[t] = (p[PW] - p[-PW]) * a.inv_dy;
        code[t] = theta_class(gx[t], gy[t], th[t]);
        if (a.wide_angles)  // uniform: some angle may lie beyond the reduced range
            kg_sincos(a.aniso * (th[t] - a.theta0), &sn[t], &cs[t]);
        else
            kg_sincos_reduced(a.aniso * (th[t] - a.theta0), &sn[t], &cs[t]);
        eps[t] = a.eps_bar * ((R)1.0 + a.delta * cs[t]);
        epsd[t] = a.neg_ebar_j_delta * sn[t];
        const R ls = (lp[t] + a.K * lT[t]) * a.dt_tau;
        sm.E2[k] = eps[t] * eps[t];
        sm.F[k] = eps[t] * epsd[t];
        sm.GX[k] = gx[t];
        sm.GY[k] = gy[t];
        sm.LS[k] = ghost[t] ? -ls : ls;
        sm.LT[k] = lT[t];
        lp[t] = ls;
    }
    if (a.noise_a != (R)0)  // one Philox block per lane, the last waves first
        for (int l = ANT - 1 - tid; l < ON / 4; l += ANT) {
            const int r = l / (AX / 4), g = l - r * (AX / 4);
            const u32x4 w = philox4x32_10(
                u32x4{(uint32_t)(x0 / 4 + g), (uint32_t)(y0 + r), step, a.instance}, a.key0,
                a.key1);
            R *x = &sm.X[4 * l];
            x[0] = noise_from_word<R>(w.x);
            x[1] = noise_from_word<R>(w.y);
            x[2] = noise_from_word<R>(w.z);
            x[3] = noise_from_word<R>(w.w);
        }
    __syncthreads();

    // ---- reverse of pass 2 on the tile -----------------------------------
    // v: the parameter sums, without the factors the host applies (tau: -1 /
    // tau, alpha: 1 / pi, eps_bar: 1 / eps_bar)
    double v[NPAR] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    R lphi_loc = (R)0, lT_loc = (R)0;
    if (own) {
        const int q = (rw + 2) * QW + cw + 2;
        const R *e2 = &sm.E2[q], *F = &sm.F[q], *X = &sm.GX[q], *Y = &sm.GY[q];
        const R *p = &sm.P[(rw + 3) * PW + cw + 3];
        const R gEx = (e2[1] - e2[-1]) * a.inv_dx, gEy = (e2[QW] - e2[-QW]) * a.inv_dy;
        const R t1 = (F[QW] * X[QW] - F[-QW] * X[-QW]) * a.inv_dy;
        const R t2 = -(F[1] * Y[1] - F[-1] * Y[-1]) * a.inv_dx;
        const R t3 = gEx * X[0] + gEy * Y[0];
        const R phi = p[0], T = Tc;
        const R u = a.gamma * (a.teq - T);
        const R atn = kg_atan(u);
        const R chi = a.noise_a != (R)0 ? sm.X[tid] : (R)0;
        const R qv = phi - (R)0.5 + a.alpha_pi * atn + a.noise_a * chi;
        const R w1 = phi * ((R)1.0 - phi);
        const R s = t1 + t2 + e2[0] * (lap9(p, PW) * a.inv_3dx2) + t3 + w1 * qv;
        const R ls = sm.LS[q], l1 = sm.LT[q];
        const R dm = w1 * a.alpha_pi / ((R)1.0 + u * u);  // w1 dm/du
        const double lsd = (double)ls;
        v[P_TAU] += lsd * (double)s;
        v[P_K] += (double)l1 * (double)(s * a.dt_tau);
        v[P_ALPHA] += lsd * (double)(w1 * atn);
        v[P_GAMMA] += lsd * (double)(dm * (a.teq - T));
        v[P_TEQ] += lsd * (double)(dm * a.gamma);
        v[P_NOISE] += lsd * (double)(w1 * chi);
        // phi enters phi' directly (coefficient 1) and through s; T' = T + lapT dt
        // + K s dt/tau has no other phi dependence (its K lT' is inside ls)
        lphi_loc = lp1 + ls * (((R)1.0 - (R)2.0 * phi) * qv + w1);
        lT_loc = l1 - ls * dm * a.gamma;
    }

    // ---- reverse of pass 1 on the 1-cell halo ----------------------------
    R lgx[TQ], lgy[TQ], le[TQ];
#pragma unroll
    for (int t = 0; t < TQ; ++t) {
        const int k = tid + t * ANT, r = k / QW, c = k - r * QW;
        if (k >= QN || r < 1 || r > AY + 2 || c < 1 || c > AX + 2)
            continue;
        const int q = ctr[t];
        const R *L = &sm.LS[q], *X = &sm.GX[q], *Y = &sm.GY[q], *e2 = &sm.E2[q];
        const R ls = lp[t], lap = lap9(&sm.P[(q / QW + 1) * PW + q % QW + 1], PW) * a.inv_3dx2;
        R le2 = ls * lap;
        le2 += L[-1] * X[-1] * a.inv_dx;
        le2 -= L[1] * X[1] * a.inv_dx;
        le2 += L[-QW] * Y[-QW] * a.inv_dy;
        le2 -= L[QW] * Y[QW] * a.inv_dy;
        const R lA = (L[-QW] - L[QW]) * a.inv_dy, lB = (L[1] - L[-1]) * a.inv_dx;
        const R gEx = (e2[1] - e2[-1]) * a.inv_dx, gEy = (e2[QW] - e2[-QW]) * a.inv_dy;
        const R F = eps[t] * epsd[t];
        const R epsd_th = a.neg_ebar_j_delta * a.aniso * cs[t];  // d eps' / d theta
        const R F_th = epsd[t] * epsd[t] + eps[t] * epsd_th;
        const R G = lA * gx[t] + lB * gy[t];
        const R lt = le2 * (R)2.0 * eps[t] * epsd[t] + G * F_th + lth[t];
        R lx = lA * F + ls * gEx, ly = lB * F + ls * gEy;
        if (code[t] == 1) {
            const R g2 = gx[t] * gx[t] + gy[t] * gy[t];
            lx += lt * (-gy[t] / g2);
            ly += lt * (gx[t] / g2);
        }
        lgx[t] = ghost[t] ? -lx : lx;
        lgy[t] = ghost[t] ? -ly : ly;
        le[t] = ls * (eps[t] * eps[t]);
        const int ux = x0 - 2 + c, uy = y0 - 2 + r;
        if (r >= 2 && r < AY + 2 && c >= 2 && c < AX + 2 && ux < nx && uy < ny) {
            io.lth0[m.off + (size_t)uy * nx + ux] = code[t] == 0 ? lt : (R)0;
            const R de_dd = a.eps_bar * cs[t], ded_dd = -a.eps_bar * a.aniso * sn[t];
            v[P_DELTA] += (double)(le2 * (R)2.0 * eps[t] * de_dd) +
                          (double)(G * (de_dd * epsd[t] + eps[t] * ded_dd));
            v[P_EPS_BAR] += (double)(le2 * (R)2.0 * eps[t] * eps[t]) + (double)(G * (R)2.0 * F);
            v[P_THETA0] -= (double)(le2 * (R)2.0 * eps[t] * epsd[t]) + (double)(G * F_th);
        }
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < TQ; ++t) {
        const int k = tid + t * ANT, r = k / QW, c = k - r * QW;
        if (k >= QN || r < 1 || r > AY + 2 || c < 1 || c > AX + 2)
            continue;
        sm.GX[k] = lgx[t];
        sm.GY[k] = lgy[t];
        sm.E2[k] = le[t];
    }
#pragma unroll
    for (int p = 0; p < NPAR; ++p) {
        const double x = row_sum(v[p]);
        if ((tid & 15) == 0)
            sm.red[p][tid >> 4] = x;
    }
    __syncthreads();

    // ---- gather of the input adjoints ------------------------------------
    if (own) {
        const int q = (rw + 2) * QW + cw + 2;
        R l = lphi_loc;
        l += sm.GX[q - 1] * a.inv_dx;
        l -= sm.GX[q + 1] * a.inv_dx;
        l += sm.GY[q - QW] * a.inv_dy;
        l -= sm.GY[q + QW] * a.inv_dy;
        l += lap9(&sm.E2[q], QW) * a.inv_3dx2;
        io.lphi0[oo] = l;
        io.lT0[oo] = lT_loc + lap9(&sm.LT[q], QW) * a.inv_3dx2 * a.dt;
    }
    if (tid < 16 * NPAR) {
        double x = 0.0;
#pragma unroll
        for (int g = 0; g < ANT / 16; g += 16)
            if (g + (tid & 15) < ANT / 16)
                x += sm.red[tid >> 4][g + (tid & 15)];
        x = row_sum(x);
        if (adder)
            *sum = before + x;
    }
}

// tiles[b] = (member, x0, y0, accumulator slot), member < 0: none
template <typename R, bool ASK>
__global__ __launch_bounds__(ANT) void k_adj_step(const AdjMember<R> *__restrict__ members,
                                                    const int4 *__restrict__ tiles, AdjIO<R> io,
                                                    double *__restrict__ acc, int nslots,
                                                    uint32_t step, int first)
{
    __shared__ AdjSmem<R> sm;
    const int4 d = tiles[blockIdx.x];
    if (d.x < 0)
        return;
    const AdjMember<R> m = members[d.x];
    if (m.a.boundary == 1)
        adj_tile<R, 1, ASK>(m, io, d.y, d.z, step, acc, nslots, d.w, first != 0, sm);
    else
        adj_tile<R, 0, ASK>(m, io, d.y, d.z, step, acc, nslots, d.w, first != 0, sm);
}

// The same for a single grid: its parameters travel with the launch and the
// tile follows from the block (the order of the table), which saves a block
// two dependent loads before its first one.
template <typename R, bool ASK>
__global__ __launch_bounds__(ANT) void k_adj_step_one(AdjMember<R> m, AdjIO<R> io,
                                                      double *__restrict__ acc, int nslots,
                                                      int first)
{
    __shared__ AdjSmem<R> sm;
    const int slot = (int)strip_tile(blockIdx.x);
    if (slot >= nslots)
        return;
    const int tiles_x = (m.a.nx + AX - 1) / AX;
    const int x0 = slot % tiles_x * AX, y0 = slot / tiles_x * AY;
    if (m.a.boundary == 1)
        adj_tile<R, 1, ASK>(m, io, x0, y0, m.a.step, acc, nslots, slot, first != 0, sm);
    else
        adj_tile<R, 0, ASK>(m, io, x0, y0, m.a.step, acc, nslots, slot, first != 0, sm);
}

// Loss of each tile = sum (phi - target)^2 in FP64; lphi = 2 (phi - target),
// lT = ltheta = 0.
constexpr int SEED_THREADS = 256;
template <typename R>
__global__ __launch_bounds__(SEED_THREADS) void k_adj_seed(
    const AdjMember<R> *__restrict__ members, const int4 *__restrict__ tiles, const R *phi,
    const R *target, R *lphi, R *lT, R *lth, double *loss, uint32_t *zero, uint32_t *zero_other)
{
    const int4 d = tiles[blockIdx.x];
    if (d.x < 0)
        return;
    const size_t off = members[d.x].off;
    const int nx = members[d.x].a.nx, ny = members[d.x].a.ny;
    double s = 0.0;
    for (int k = threadIdx.x; k < ON; k += SEED_THREADS) {
        const int i = d.y + k % AX, j = d.z + k / AX;
        if (i >= nx || j >= ny)
            continue;
        const size_t o = off + (size_t)j * nx + i;
        const R e = phi[o] - target[o];
        s += (double)e * (double)e;
        lphi[o] = (R)2.0 * e;
        lT[o] = (R)0;
        lth[o] = (R)0;
    }
    __shared__ double sh[SEED_THREADS / 16];
    s = row_sum(s);
    if ((threadIdx.x & 15) == 0)
        sh[threadIdx.x >> 4] = s;
    __syncthreads();
    if (threadIdx.x < 16) {
        s = row_sum(sh[threadIdx.x]);
        if (threadIdx.x == 0) {
            loss[d.w] = s;
            zero[d.w] = s == 0.0 ? 1u : 0u;  // (squares of differences: NaN is not zero)
            zero_other[d.w] = 0u;
        }
    }
}

// Block (m, p): member m's loss (p = 0) or parameter sum p - 1 over its tiles'
// slots [first[m], first[m + 1]), to out[m * (NPAR + 1) + p].
__global__ __launch_bounds__(SEED_THREADS) void k_adj_total(const int *__restrict__ first,
                                                            const double *__restrict__ acc,
                                                            const double *__restrict__ loss,
                                                            int nslots, double *__restrict__ out)
{
    const int lo = first[blockIdx.x], hi = first[blockIdx.x + 1], p = blockIdx.y;
    __shared__ double sh[SEED_THREADS / 16];
    const double *src = p == 0 ? loss : acc + (size_t)(p - 1) * nslots;
    double s = 0.0;
    for (int k = lo + threadIdx.x; k < hi; k += SEED_THREADS)
        s += src[k];
    s = row_sum(s);
    if ((threadIdx.x & 15) == 0)
        sh[threadIdx.x >> 4] = s;
    __syncthreads();
    if (threadIdx.x < 16) {
        s = row_sum(sh[threadIdx.x]);
        if (threadIdx.x == 0)
            out[(size_t)blockIdx.x * (NPAR + 1) + p] = s;
    }
}

}  // namespace

struct AdjointWork {
    size_t total = 0;        // elements per field buffer
    size_t esize = 0;
    int ckpt_cap = 0, seg_cap = 0, nmembers = 0;
    int nslots = 0, nblocks = 0;  // tiles, and tile table entries
    char *ckpt = nullptr;    // ckpt_cap states of 3 fields
    char *seg = nullptr;     // seg_cap + 1 states of 3 fields
    char *lam = nullptr;     // 2 x (lphi, lT, ltheta)
    char *target = nullptr;
    double *acc = nullptr;   // NPAR x nslots
    double *loss = nullptr;  // nslots
    uint32_t *zero = nullptr; // 2 x nslots: AdjIO's words of the two adjoint buffers
    double *out = nullptr;   // nmembers x (NPAR + 1)
    void *members = nullptr; // AdjMember<R>[nmembers]
    int4 *tiles = nullptr;
    int *first = nullptr;    // nmembers + 1: a member's first slot
};

void free_adjoint(AdjointWork *w)
{
    if (!w)
        return;
    void *p[] = {w->ckpt, w->seg, w->lam, w->target, w->acc, w->loss, w->zero, w->out, w->members,
                 w->tiles, w->first};
    for (void *q : p)
        if (q)
            (void)hipFree(q);
    delete w;
}

namespace {

// What adjoint_core needs of a single grid or a batch.
template <typename R>
struct AdjJob {
    hipStream_t stream;
    size_t total;                       // elements per field buffer
    std::vector<int> nx, ny;
    std::vector<size_t> off;
    std::vector<kg_params> params;
    std::vector<int> wide;              // StepArgs::wide_angles of each member
    uint64_t s0;                        // noise counter of the first step
    const void *const *targets;         // host fields of the members
    void *const *d_T0, *const *d_phi0;  // host results, null entries: not wanted
    std::function<void(R *cur[3])> current;  // the job's own current buffers
    std::function<int(int n)> forward;       // n steps on them
    std::function<void(int n)> skip;         // count n steps taken elsewhere
    // steps from state `in` to the states that follow it (3 * total elements
    // apart): up to n of them, or a negative status
    std::function<int(R *const *in, R *const *out, uint32_t step, int n)> steps;
};

// Whether the reverse steps keep and ask for the words of all-zero tiles: the
// adjoint starts where phi and the target differ and spreads 2 cells a step,
// so most of a large grid is zero for many steps (FP32, whole adjoints: 24
// members of 128^2 .. 512^2, 100 steps, 8.25 -> 7.2 ms; 1500 x 1400, 50 steps,
// 3.28 -> 2.69).  A launch that fits the chip at once only waits a round trip
// longer (190 x 133 FP64 1.41 -> 1.46), and in FP64, where tails underflow 10
// times as far out, little is zero (the 24 members 16.2 -> 16.6).
template <typename R>
bool asks_zero(int ntiles)
{
    return sizeof(R) == 4 && ntiles > 2048;
}

template <typename R, bool ASK>
hipError_t launch_reverse_as(const AdjointWork &w, const std::vector<AdjMember<R>> &mem,
                             const AdjIO<R> &io, uint32_t step, bool first, hipStream_t s)
{
    if (mem.size() == 1) {
        AdjMember<R> m = mem[0];
        m.a.step = step;
        hipLaunchKernelGGL((k_adj_step_one<R, ASK>), dim3(w.nblocks), dim3(ANT), 0, s, m,
                           io, w.acc, w.nslots, first ? 1 : 0);
    } else {
        hipLaunchKernelGGL((k_adj_step<R, ASK>), dim3(w.nblocks), dim3(ANT), 0, s,
                           static_cast<const AdjMember<R> *>(w.members), w.tiles, io, w.acc,
                           w.nslots, step, first ? 1 : 0);
    }
    return hipGetLastError();
}

template <typename R>
hipError_t launch_reverse(const AdjointWork &w, const std::vector<AdjMember<R>> &mem,
                          const AdjIO<R> &io, uint32_t step, bool first, hipStream_t s)
{
    if constexpr (sizeof(R) == 4)
        if (asks_zero<R>(w.nslots))
            return launch_reverse_as<R, true>(w, mem, io, step, first, s);
    return launch_reverse_as<R, false>(w, mem, io, step, first, s);
}

// Buffers and tile table of the job, sized for nckpt checkpoints and segments
// of seglen steps; reused while large enough (a handle's grids never change).
template <typename R>
int ensure_work(AdjointWork *&w, const AdjJob<R> &job, int nckpt, int seglen)
{
    const size_t fb = job.total * sizeof(R);
    const int M = (int)job.nx.size();
    if (w && (w->ckpt_cap < nckpt || w->seg_cap < seglen)) {
        free_adjoint(w);
        w = nullptr;
    }
    if (w)
        return KG_OK;
    // tiles member by member, dealt in strips
    std::vector<int4> t;
    std::vector<int> first(1, 0);
    for (int m = 0; m < M; ++m) {
        for (int y = 0; y < job.ny[m]; y += AY)
            for (int x = 0; x < job.nx[m]; x += AX)
                t.push_back(make_int4(m, x, y, (int)t.size()));
        first.push_back((int)t.size());
    }
    const int n = (int)t.size();
    std::vector<int4> dealt(strip_blocks(t.size()), make_int4(-1, 0, 0, 0));
    for (unsigned b = 0; b < dealt.size(); ++b)
        if (strip_tile(b) < t.size())
            dealt[b] = t[strip_tile(b)];
    w = new AdjointWork();
    w->total = job.total;
    w->esize = sizeof(R);
    w->ckpt_cap = nckpt;
    w->seg_cap = seglen;
    w->nmembers = M;
    w->nslots = n;
    w->nblocks = (int)dealt.size();
    bool ok = (nckpt == 0 || hipMalloc(&w->ckpt, 3 * fb * (size_t)nckpt) == hipSuccess) &&
              hipMalloc(&w->seg, 3 * fb * (size_t)(seglen + 1)) == hipSuccess &&
              hipMalloc(&w->lam, 6 * fb) == hipSuccess && hipMalloc(&w->target, fb) == hipSuccess &&
              hipMalloc(&w->acc, (size_t)NPAR * n * sizeof(double)) == hipSuccess &&
              hipMalloc(&w->loss, (size_t)n * sizeof(double)) == hipSuccess &&
              hipMalloc(&w->zero, 2 * (size_t)n * sizeof(uint32_t)) == hipSuccess &&
              hipMalloc(&w->out, (size_t)M * (NPAR + 1) * sizeof(double)) == hipSuccess &&
              hipMalloc(&w->members, (size_t)M * sizeof(AdjMember<R>)) == hipSuccess &&
              hipMalloc(&w->tiles, dealt.size() * sizeof(int4)) == hipSuccess &&
              hipMalloc(&w->first, first.size() * sizeof(int)) == hipSuccess;
    hipError_t e = hipSuccess;
    if (ok) {
        e = hipMemcpyAsync(w->tiles, dealt.data(), dealt.size() * sizeof(int4),
                           hipMemcpyHostToDevice, job.stream);
        if (e == hipSuccess)
            e = hipMemcpyAsync(w->first, first.data(), first.size() * sizeof(int),
                               hipMemcpyHostToDevice, job.stream);
        if (e == hipSuccess)
            e = hipStreamSynchronize(job.stream);
    }
    if (!ok || e != hipSuccess) {
        free_adjoint(w);
        w = nullptr;
        return ok ? hip_fail(e, "adjoint tile table upload")
                  : fail(KG_ERR_OUT_OF_MEMORY, "hipMalloc of the adjoint buffers failed");
    }
    return KG_OK;
}

template <typename R>
int adjoint_core(AdjJob<R> &job, AdjointWork *&work, int nsteps, int every,
                 std::vector<kg_grads> &grads)
{
    const int M = (int)job.nx.size();
    const size_t fb = job.total * sizeof(R);
    const int nseg = (nsteps + every - 1) / every;
    // the last segment is stepped into the segment's buffers at once, so it
    // needs neither a checkpoint nor a second pass
    if (int rc = ensure_work(work, job, nseg - 1, every))
        return rc;
    AdjointWork &w = *work;
    const hipStream_t s = job.stream;
    std::vector<AdjMember<R>> mem(M);
    for (int m = 0; m < M; ++m) {
        mem[m].a = make_args<R>(job.params[m], job.nx[m], job.ny[m]);
        mem[m].a.wide_angles = job.wide[m];
        mem[m].off = job.off[m];
    }
    KG_HIP(hipMemcpyAsync(w.members, mem.data(), M * sizeof(AdjMember<R>), hipMemcpyHostToDevice, s));
    auto st = [&](char *base, int k, int f) { return reinterpret_cast<R *>(base + (3 * (size_t)k + f) * fb); };
    R *tgt = reinterpret_cast<R *>(w.target);
    auto bytes = [&](int m) { return (size_t)job.nx[m] * job.ny[m] * sizeof(R); };
    for (int m = 0; m < M; ++m)
        KG_HIP(hipMemcpyAsync(tgt + job.off[m], job.targets[m], bytes(m), hipMemcpyHostToDevice, s));

    // forward with checkpoints
    R *cur[3];
    auto copy_state = [&](char *base, int k) -> int {  // current state -> slot k
        job.current(cur);
        for (int f = 0; f < 3; ++f)
            KG_HIP(hipMemcpyAsync(st(base, k, f), cur[f], fb, hipMemcpyDeviceToDevice, s));
        return KG_OK;
    };
    auto fill_segment = [&](int k, int len) -> int {  // states 1 .. len from state 0
        for (int i = 0; i < len;) {
            R *in[3] = {st(w.seg, i, 0), st(w.seg, i, 1), st(w.seg, i, 2)};
            R *out[3] = {st(w.seg, i + 1, 0), st(w.seg, i + 1, 1), st(w.seg, i + 1, 2)};
            const int n = job.steps(in, out, (uint32_t)(job.s0 + (uint64_t)k * every + i), len - i);
            if (n < 0)
                return n;
            i += n;
        }
        return KG_OK;
    };
    for (int k = 0; k < nseg - 1; ++k) {
        if (int rc = copy_state(w.ckpt, k))
            return rc;
        if (int rc = job.forward(every))
            return rc;
    }
    const int last = nsteps - (nseg - 1) * every;
    if (int rc = copy_state(w.seg, 0))
        return rc;
    if (int rc = fill_segment(nseg - 1, last))
        return rc;
    job.skip(last);
    job.current(cur);
    for (int f = 0; f < 3; ++f)
        KG_HIP(hipMemcpyAsync(cur[f], st(w.seg, last, f), fb, hipMemcpyDeviceToDevice, s));

    // loss and the seed adjoint
    R *lam[2][3];
    for (int b = 0; b < 2; ++b)
        for (int f = 0; f < 3; ++f)
            lam[b][f] = reinterpret_cast<R *>(w.lam + (3 * (size_t)b + f) * fb);
    hipLaunchKernelGGL((k_adj_seed<R>), dim3(w.nblocks), dim3(SEED_THREADS), 0, s,
                       static_cast<const AdjMember<R> *>(w.members), w.tiles,
                       (const R *)st(w.seg, last, 0), (const R *)tgt, lam[0][0], lam[0][1],
                       lam[0][2], w.loss, w.zero, w.zero + w.nslots);
    KG_HIP(hipGetLastError());

    int lc = 0;
    for (int k = nseg - 1; k >= 0; --k) {
        const int len = std::min(every, nsteps - k * every);
        if (k < nseg - 1) {  // recompute the segment's states
            for (int f = 0; f < 3; ++f)
                KG_HIP(hipMemcpyAsync(st(w.seg, 0, f), st(w.ckpt, k, f), fb,
                                      hipMemcpyDeviceToDevice, s));
            if (int rc = fill_segment(k, len))
                return rc;
        }
        for (int i = len - 1; i >= 0; --i) {
            const AdjIO<R> io{st(w.seg, i, 0), st(w.seg, i, 1), st(w.seg, i, 2),
                              lam[lc][0], lam[lc][1], lam[lc][2],
                              lam[lc ^ 1][0], lam[lc ^ 1][1], lam[lc ^ 1][2],
                              w.zero + (size_t)lc * w.nslots, w.zero + (size_t)(lc ^ 1) * w.nslots};
            const hipError_t e =
                launch_reverse<R>(w, mem, io, (uint32_t)(job.s0 + (uint64_t)k * every + i),
                                  k == nseg - 1 && i == len - 1, s);
            if (e != hipSuccess)
                return hip_fail(e, "adjoint step launch");
            lc ^= 1;
        }
    }
    hipLaunchKernelGGL(k_adj_total, dim3(M, NPAR + 1), dim3(SEED_THREADS), 0, s, w.first, w.acc, w.loss,
                       w.nslots, w.out);
    KG_HIP(hipGetLastError());
    std::vector<double> out((size_t)M * (NPAR + 1));
    std::vector<HostPiece> back{{out.data(), w.out, out.size() * sizeof(double)}};
    for (int m = 0; m < M; ++m) {
        if (job.d_T0 && job.d_T0[m])
            back.push_back({job.d_T0[m], lam[lc][1] + job.off[m], bytes(m)});
        if (job.d_phi0 && job.d_phi0[m])
            back.push_back({job.d_phi0[m], lam[lc][0] + job.off[m], bytes(m)});
    }
    KG_HIP(copy_to_host(s, back.data(), (int)back.size()));
    grads.assign(M, kg_grads{});
    for (int m = 0; m < M; ++m) {
        const double *o = &out[(size_t)m * (NPAR + 1)], *v = o + 1;
        kg_grads &g = grads[m];
        g.loss = o[0];
        g.d_tau = -v[P_TAU] / (double)(R)job.params[m].tau;
        g.d_eps_bar = v[P_EPS_BAR] / (double)(R)job.params[m].eps_bar;
        g.d_K = v[P_K];
        g.d_delta = v[P_DELTA];
        g.d_theta0 = v[P_THETA0];
        g.d_alpha = v[P_ALPHA] / (double)(sizeof(R) == 4 ? (R)3.14159274f : (R)3.14159265358979323846);
        g.d_gamma = v[P_GAMMA];
        g.d_teq = v[P_TEQ];
        g.d_noise_a = v[P_NOISE];
    }
    return KG_OK;
}

template <typename R>
int adjoint_single(kg_solver_s &h, int nsteps, int every, const void *target, kg_grads *out,
                   void *d_T0, void *d_phi0)
{
    AdjJob<R> job;
    job.stream = h.stream;
    job.total = h.cells();
    job.nx = {h.nx};
    job.ny = {h.ny};
    job.off = {0};
    job.params = {h.params};
    job.wide = {wide_angles(h.params, h.theta_given)};
    job.s0 = h.steps;
    job.targets = &target;
    job.d_T0 = &d_T0;
    job.d_phi0 = &d_phi0;
    // the forward steps below run without tile status: it no longer describes
    // the handle's buffers afterwards
    h.stat_valid = false;
    StepArgs<R> base = make_args<R>(h.params, h.nx, h.ny);
    base.wide_angles = job.wide[0];
    job.current = [&](R *cur[3]) {
        cur[0] = static_cast<R *>(h.phi[h.cur]);
        cur[1] = static_cast<R *>(h.T[h.cur]);
        cur[2] = static_cast<R *>(h.theta);
    };
    job.forward = [&](int n) -> int {
        for (int i = 0; i < n;) {
            StepArgs<R> a = base;
            a.phi_in = static_cast<const R *>(h.phi[h.cur]);
            a.T_in = static_cast<const R *>(h.T[h.cur]);
            a.phi_out = static_cast<R *>(h.phi[h.cur ^ 1]);
            a.T_out = static_cast<R *>(h.T[h.cur ^ 1]);
            a.theta = static_cast<R *>(h.theta);
            if (h.theta_alt && n - i >= MULTI_STEPS) {
                KG_HIP(step_multi<R>(h, a));
                i += MULTI_STEPS;
                continue;
            }
            a.step = (uint32_t)h.steps;
            KG_HIP(launch_step_fused<R>(a, h.stream));
            h.cur ^= 1;
            h.steps += 1;
            ++i;
        }
        return KG_OK;
    };
    job.skip = [&](int n) { h.steps += (uint64_t)n; };
    // the small tiles take the old angles from another buffer; the 64 x 30
    // tiles update theta in place, on a copy
    const bool small = small_shape(h.nx, h.ny, sizeof(R)) != 0;
    job.steps = [&, small](R *const *in, R *const *o, uint32_t step, int n) -> int {
        StepArgs<R> a = base;
        a.phi_in = in[0];
        a.T_in = in[1];
        a.phi_out = o[0];
        a.T_out = o[1];
        a.theta = o[2];
        a.step = step;
        if (h.theta_alt && n >= MULTI_STEPS) {
            a.theta_in = in[2];
            KG_HIP(launch_step_multi<R>(a, 3 * job.total, h.stream));
            return MULTI_STEPS;
        }
        if (small)
            a.theta_in = in[2];
        else
            KG_HIP(hipMemcpyAsync(o[2], in[2], h.field_bytes(), hipMemcpyDeviceToDevice, h.stream));
        KG_HIP(launch_step_fused<R>(a, h.stream));
        return 1;
    };
    std::vector<kg_grads> g;
    if (int rc = adjoint_core<R>(job, h.adj, nsteps, every, g))
        return rc;
    *out = g[0];
    return KG_OK;
}

template <typename R>
int adjoint_batch(kg_batch_s &b, int nsteps, int every, const void *const *targets, kg_grads *out,
                  void *const *d_T0)
{
    AdjJob<R> job;
    job.stream = b.stream;
    job.total = b.total;
    job.nx = b.nx;
    job.ny = b.ny;
    job.off = b.off;
    job.params = b.params;
    for (int m = 0; m < b.count; ++m)
        job.wide.push_back(wide_angles(b.params[m], b.theta_given[m]));
    job.s0 = b.steps;
    job.targets = targets;
    job.d_T0 = d_T0;
    job.d_phi0 = nullptr;
    job.current = [&](R *cur[3]) {
        cur[0] = static_cast<R *>(b.phi[b.cur()]);
        cur[1] = static_cast<R *>(b.T[b.cur()]);
        cur[2] = static_cast<R *>(b.theta);
    };
    job.forward = [&](int n) -> int { return kg_batch_step(&b, n); };
    job.skip = [&](int n) { b.steps += (uint64_t)n; };
    job.steps = [&](R *const *in, R *const *o, uint32_t step, int n) -> int {
        const int steps = multi_shape_steps(b.multi_shape);
        if (b.multi_shape != 0 && n >= steps) {
            KG_HIP(batch_multi<R>(b, MultiIO<R>{in[0], in[1], in[2], o[0], o[1], o[2]}, step,
                                  3 * b.total));
            return steps;
        }
        KG_HIP(launch_step_batch_direct<R>(static_cast<const AdjMember<R> *>(b.adj->members),
                                           b.tiles, b.ntiles, in[0], in[1], in[2], o[0], o[1], o[2],
                                           step, b.stream));
        return 1;
    };
    std::vector<kg_grads> g;
    const int rc = adjoint_core<R>(job, b.adj, nsteps, every, g);
    b.stat_valid = false;  // the last segment's states were copied into the batch's buffers
    if (rc)
        return rc;
    for (int m = 0; m < b.count; ++m)
        out[m] = g[m];
    return KG_OK;
}

}  // namespace

}  // namespace kg

extern "C" int kg_batch_adjoint(kg_batch b, int nsteps, int checkpoint_every,
                                const void *const *targets, kg_grads *out, void *const *d_T0)
{
    if (!b)
        return kg::fail(KG_ERR_INVALID_ARGUMENT, "null batch");
    if (!targets || !out)
        return kg::fail(KG_ERR_INVALID_ARGUMENT, "null targets or output");
    for (int m = 0; m < b->count; ++m)
        if (!targets[m])
            return kg::fail(KG_ERR_INVALID_ARGUMENT, "null target of a member");
    if (nsteps < 1 || checkpoint_every < 1)
        return kg::fail(KG_ERR_INVALID_ARGUMENT, "nsteps and checkpoint_every must be >= 1");
    KG_HIP(hipSetDevice(b->device));
    const int every = std::min(checkpoint_every, nsteps);
    return b->precision == KG_F64
               ? kg::adjoint_batch<double>(*b, nsteps, every, targets, out, d_T0)
               : kg::adjoint_batch<float>(*b, nsteps, every, targets, out, d_T0);
}

extern "C" int kg_adjoint(kg_handle h, int nsteps, int checkpoint_every, const void *target,
                          size_t bytes, kg_grads *out, void *d_T0, void *d_phi0)
{
    if (!h)
        return kg::fail(KG_ERR_INVALID_ARGUMENT, "null handle");
    if (!target || !out)
        return kg::fail(KG_ERR_INVALID_ARGUMENT, "null target or output");
    if (nsteps < 1 || checkpoint_every < 1)
        return kg::fail(KG_ERR_INVALID_ARGUMENT, "nsteps and checkpoint_every must be >= 1");
    if (bytes != h->field_bytes())
        return kg::fail(KG_ERR_SIZE, "target size does not match the field size");
    KG_HIP(hipSetDevice(h->device));
    const int every = std::min(checkpoint_every, nsteps);
    return h->precision == KG_F64
               ? kg::adjoint_single<double>(*h, nsteps, every, target, out, d_T0, d_phi0)
               : kg::adjoint_single<float>(*h, nsteps, every, target, out, d_T0, d_phi0);
}

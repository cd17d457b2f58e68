// HIP element-loop RHS of the MI355X ADS step in 3D (gfx950), variant 4 in one launch: the
// integrals of compute_rhs (validation.hpp:95-119) with every one-dimensional contraction
// shared by the elements that need it.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "adsg_device.hpp"

namespace adsg {

namespace {

// ------------------------------------------------------------------------------------
// Sum factorisation over a column of elements instead of per element. A workgroup owns a
// tile of TX x 4 elements in x and y and marches along z; a wave owns one element row along
// x, a lane one x Gauss point (qx) of it with all M = P + 1 y Gauss points. Per DOF plane:
//  U  the wave's M rows of coefficients, staged in LDS, contracted along x (value, derivative),
//  Y  along y for its Gauss points: u, u_y, u_x, kept in registers for the last M planes,
//  Z  for the element whose last plane this is: along z, the integrand at the Gauss points,
//     the z-transposed sums, kept in registers for the M planes the element touches,
//  T  the element's first plane is complete: y transposed, exchanged between the lanes of an
//     x element through LDS, x transposed (S), the element contributions of the M rows added
//     to the tile's block in LDS.
// After M planes and one barrier the rows that neighbouring waves share are summed in a fixed
// order and written: entries the tile owns to the rhs, the others to the spill arrays of the
// one-launch tiling (adsg_rhs.hip), which k_rhs_fixup adds. The x and y contractions run once
// per plane and row instead of once per element, M^2 and M times less: 576 FP64 operations
// per lane and plane at p = 3 without a mass term, 36 per Gauss point column; the per-element
// kernel spends 4768 multiply-adds per element, this one about 2400.
// Bound: FP64 issue (1.85 ns per wave instruction and SIMD, dependent or not). The element
// pass of 192^3, p = 3, FP64 without a mass term went from 2197 to 893 us (FP32 from 1197 us
// on the matrix cores to 689), 128^3, p = 2 from 165 to 136 us (FP32 98 to 103, with shorter
// sweeps after it than the kernels that were replaced had), with a k field (70 x 50 x 61, p = 2)
// from 154 us in colour launches to 34. Measured on the way: lanes over
// element pairs of y Gauss points at twice the waves (more instructions, 1.5x slower); the z
// tables as DPP broadcast operands instead of scalar registers (more registers: spills); the
// x contraction one plane ahead and the block write spread over the planes (registers again:
// 3 to 20 % slower). What is left is the register file: at p = 3 FP64 the 256 registers of 2
// waves per SIMD hold all but 39 to 72 of the values (scratch), and 2 or 3 waves hide little of
// the LDS and scalar-load latency.
// ------------------------------------------------------------------------------------
template <int P>
struct march {
    static constexpr int M = P + 1;
    // elements of a wave along x: one lane per x Gauss point, and (p <= 2) the M rows of
    // TX + P DOFs that a wave stages and writes per plane fit its 64 lanes too
    static constexpr int TX = P == 1 ? 31 : P == 2 ? 19 : 16;
    static constexpr int BX = TX + P;
    static constexpr int NL = (M * BX + 63) / 64;  // passes of 64 lanes over M rows of BX
    static constexpr int SX = 64 / M + 1 + 2 * P;  // padded row of the x sums, every lane's element in it
    static constexpr int RP = 64 / BX;             // rows of BX DOFs per wave in the block write
};
// element rows (waves) per workgroup: one wave per SIMD (five or six waves measured 1.7x
// slower: the SIMD with two of them sets the pace between the barriers; eight 1.2x)
constexpr int kMarchRows = 4;
// waves per SIMD the register allocation must allow: the window of M planes and the sums of M
// planes are 6 M^2 values per lane (7 M^2 with a k field), the sums FP64 in both precisions (FP32
// at p = 3 in 3 waves: 214 registers spilled)
constexpr int march_waves(int bytes, int p, bool kfield) {
    return p == 3 ? (bytes == 8 && kfield ? 1 : 2) : bytes == 8 && p == 2 && kfield ? 2 : 3;
}

template <typename T, int P, bool KF>
struct march_lds {  // values per workgroup
    using S = march<P>;
    static constexpr int XT = 4 * S::M * 64;
    static constexpr int UB = (KF ? 2 : 1) * S::NL * 64, KB = 2 * S::M * 64, SB = S::M * S::M * S::SX;
    static constexpr int PLANE = (kMarchRows + P) * S::M * S::BX;  // doubles: a plane of the block
    static constexpr size_t bytes() {
        return (XT + kMarchRows * (UB + KB + SB)) * sizeof(T) + 2 * S::M * PLANE * sizeof(double);
    }
};

template <typename T>
struct march_args {
    const T* up;
    const T* kfield;
    T* rhs;
    const T* start;  // when set: rhs := scale * start + sums
    T* spill;
    const T* tab[3];  // packed tables per direction (dev_tables::pack)
    long off[8];      // spill layout (rhs_params)
    int ext[3][2];
    int n[3], el[3];  // DOFs and elements
    int ntx, nty, tz;
    T cx, cy, cz, mass, rdt, scale;
};

template <typename T>
__device__ __forceinline__ T* at(T* base, unsigned bytes) {  // a 32-bit lane offset on a uniform base
    return reinterpret_cast<T*>(reinterpret_cast<char*>(base) + bytes);
}
template <typename T>
__device__ __forceinline__ const T* at(const T* base, unsigned bytes) {
    return reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + bytes);
}

// FM: 0 the heat form (mass term), 1 with the reaction term, 2 no mass term, KF: k field
template <typename T, int P, bool KF, int FM>
__global__ __launch_bounds__((64 * kMarchRows), march_waves(sizeof(T), P, KF)) void k_rhs3_march(march_args<T> A) {
    using S = march<P>;
    using L = march_lds<T, P, KF>;
    constexpr int M = P + 1, TX = S::TX, TY = kMarchRows, BX = S::BX, NL = S::NL, SX = S::SX, RP = S::RP;
    constexpr int TAB = 4 * M * M;  // table values per element
    constexpr bool RX = FM == 1, MS = FM != 2;
    static_assert(RP * TY >= TY + P, "one pass writes a plane of the block");
    extern __shared__ double march_smem[];

    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int tz = A.tz;
    int t = xcd_contiguous(blockIdx.x, gridDim.x);
    const int tix = t % A.ntx;
    t /= A.ntx;
    const int tiy = t % A.nty, tiz = t / A.nty;
    const int ex0 = tix * TX, ey0 = tiy * TY, ez0 = tiz * tz;
    const int nact = min(TY, A.el[1] - ey0);                   // element rows of the tile
    const int nzl = min(tz, A.el[2] - ez0), npl = nzl + P;     // its elements and planes along z
    const int nx = A.n[0], ny = A.n[1];
    const long pstride = static_cast<long>(nx) * ny;

    // the tile's block, M planes in two buffers: [2][M planes][TY + P rows][M][BX], entry r of
    // row b from the wave of element row b - r (zero where there is none)
    double* part = march_smem;
    T* xt = reinterpret_cast<T*>(part + 2 * M * L::PLANE);  // [4][M][64]
    T* ub = xt + L::XT + wv * (L::UB + L::KB + L::SB);       // [M][BX] (and of the k field)
    T* kb = ub + L::UB;                                      // [2][M][64]
    T* sb = kb + L::KB;                                      // [M][M][SX]

    // x tables per lane (Gauss point q of element el): the forward rows (val, der)[q][.], and
    // the backward columns (val, der)[.][q] with the weight (and -dt*grad_x) folded in
    const int el = lane / M, q = lane % M;
    {
        const bool in = el < TX && ex0 + el < A.el[0];
        const T* tb = A.tab[0] + static_cast<long>(in ? ex0 + el : 0) * TAB;
        for (int r = wv; r < M; r += TY) {
            xt[(0 * M + r) * 64 + lane] = in ? tb[(q * 4 + 0) * M + r] : T(0);
            xt[(1 * M + r) * 64 + lane] = in ? tb[(q * 4 + 1) * M + r] : T(0);
            xt[(2 * M + r) * 64 + lane] = in ? tb[(r * 4 + 2) * M + q] : T(0);
            xt[(3 * M + r) * 64 + lane] = in ? A.cx * tb[(r * 4 + 3) * M + q] : T(0);
        }
        for (int i = lane; i < L::SB; i += 64) sb[i] = T(0);
        for (int i = threadIdx.x; i < 2 * M * L::PLANE; i += 64 * TY) part[i] = 0.0;
    }
    __syncthreads();

    // this lane's part of the M rows of BX coefficients the wave stages per plane: byte offsets
    // in the plane, clamped to the mesh (entries beyond it meet zero tables only)
    const bool act = wv < nact;
    unsigned goff[NL];
#pragma unroll
    for (int j = 0; j < NL; ++j) {
        const int l = j * 64 + lane, r = min(l / BX, M - 1), i = l % BX;
        goff[j] = (static_cast<unsigned>(min(ex0 + i, nx - 1)) +
                   static_cast<unsigned>(nx) * static_cast<unsigned>(min(ey0 + wv + r, ny - 1))) * sizeof(T);
    }
    T pre[NL], prek[KF ? NL : 1];
    auto fetch = [&](int k) {
        const long o = (ez0 + min(k, npl - 1)) * pstride;
#pragma unroll
        for (int j = 0; j < NL; ++j) {
            pre[j] = *at(A.up + o, goff[j]);
            if constexpr (KF) prek[j] = *at(A.kfield + o, goff[j]);
        }
    };

    // this lane's entry of the tile's block: row ob, column oi. Its sums go to the rhs when the
    // tile owns the DOF (kind 0), else to the spill array of the owner's offset in x and y
    // (kind dx + 2 dy; 4 more for the planes of the next tile along z), at byte offset ooff
    // of the plane
    const int oi = lane % BX, ob = wv * RP + lane / BX;
    int kind = -1;
    unsigned ooff = 0;
    if (lane < RP * BX && ob < nact + P && ex0 + oi < nx) {
        const int dx = oi >= TX && ex0 + TX < A.el[0], dy = ob >= TY && ey0 + TY < A.el[1];
        kind = dx + 2 * dy;
        const int cx = dx ? (tix + 1) * P + oi - TX : ex0 + oi, cy = dy ? (tiy + 1) * P + ob - TY : ey0 + ob;
        ooff = (cx + static_cast<unsigned>(dx ? A.ext[0][1] : A.ext[0][0]) * static_cast<unsigned>(cy)) * sizeof(T);
    }
    const bool lastz = ez0 + tz >= A.el[2];

    // LDS indices of the lane, made opaque once per plane: the addresses derived from them are
    // then formed where they are used instead of being kept in (spilled) registers
    int i_lane = lane, i_el = el, i_k = el * M, i_sw = q * SX + P + el, i_out = min(ob, TY + P - 1) * M * BX + oi;
    int i_sr[NL], i_pw[NL];
#pragma unroll
    for (int j = 0; j < NL; ++j) {
        const int l = min(j * 64 + lane, M * BX - 1), r = l / BX, i = l % BX;
        i_sr[j] = r * M * SX + P + i;
        i_pw[j] = ((wv + r) * M + r) * BX + i;
    }
    auto opaque = [&]() {
        asm volatile("" : "+v"(i_lane), "+v"(i_el), "+v"(i_k), "+v"(i_sw), "+v"(i_out));
#pragma unroll
        for (int j = 0; j < NL; ++j) asm volatile("" : "+v"(i_sr[j]), "+v"(i_pw[j]));
    };
    // FP32: the contractions take differences from the element's first coefficient (its first row,
    // its first plane), which the derivatives are made of: their rounding errors scale with the
    // variation of u over the element (the basis functions sum to 1, their derivatives to 0).
    // The sums of different elements are FP64 in both precisions.
    constexpr bool REL = sizeof(T) == sizeof(float);
    auto stage = [&]() {
#pragma unroll
        for (int j = 0; j < NL; ++j) {
            ub[j * 64 + i_lane] = pre[j];
            if constexpr (KF) ub[(NL + j) * 64 + i_lane] = prek[j];
        }
    };
    auto load_tab = [&](int k, T (&v)[M], T (&d)[M]) {
#pragma unroll
        for (int a = 0; a < M; ++a) {
            v[a] = xt[(k * M + a) * 64 + i_lane];
            d[a] = xt[((k + 1) * M + a) * 64 + i_lane];
        }
    };

    T w00[M][M], w01[M][M], w10[M][M], wk[KF ? M : 1][KF ? M : 1];  // [plane mod M][y Gauss point]
    T w0[REL ? M : 1];  // [plane mod M]: the coefficient that w00 is relative to
    double h0[M][M], hx[M][M], hy[M][M];
#pragma unroll
    for (int s = 0; s < M; ++s)
#pragma unroll
        for (int y = 0; y < M; ++y) {
            w00[s][y] = w01[s][y] = w10[s][y] = T(0);
            h0[s][y] = hx[s][y] = hy[s][y] = 0.0;
        }
    const T* ytab = A.tab[1] + static_cast<long>(ey0 + (act ? wv : 0)) * TAB;

    // the block write of the M planes from e0 on, from part buffer par
    auto write_block = [&](int par, int e0) {
        double v[M];
#pragma unroll
        for (int kk = 0; kk < M; ++kk) {
            v[kk] = 0;
#pragma unroll
            for (int r = 0; r < M; ++r) v[kk] += part[i_out + (par * M + kk) * L::PLANE + r * BX];
        }
#pragma unroll
        for (int kk = 0; kk < M; ++kk) {
            const int eo = e0 + kk;
            if (eo < 0 || eo >= npl) continue;
            const bool dz = eo >= tz && !lastz;
            if (A.start && !dz && kind == 0)
                v[kk] += static_cast<double>(A.scale * *at(A.start + (ez0 + eo) * pstride, ooff));
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                const long sz = static_cast<long>(A.ext[0][d & 1]) * A.ext[1][d >> 1];
                // selects by arithmetic: a selected address would put the arguments in scratch memory
                const long o0 = A.off[d], o4 = A.off[4 + d], m = -static_cast<long>(dz);
                const long c0 = ez0 + eo, c4 = (tiz + 1) * P + eo - tz;
                T* base = (d == 0 && !dz ? A.rhs : A.spill) + (o0 + ((o4 - o0) & m)) + sz * (c0 + ((c4 - c0) & m));
                if (kind == d) *at(base, ooff) = static_cast<T>(v[kk]);
            }
        }
    };

    int par = 0;
    const int kend = npl + P + 1;
    if (!act) {  // a row beyond the mesh: only its share of the block write
#pragma unroll 1
        for (int k0 = 0; k0 < kend; k0 += M, par ^= 1) {
            __syncthreads();
            write_block(par, k0 - P - 1);
        }
        return;
    }
    fetch(0);
    stage();
    fetch(1);
#pragma unroll 1
    for (int k0 = 0; k0 < kend; k0 += M, par ^= 1) {
#pragma unroll
        for (int kk = 0; kk < M; ++kk) {
            const int k = k0 + kk, e = k - P;  // plane k, element e = its first plane
            opaque();
            wave_lds_sync();
            T A0[M], A1[M], AK[KF ? M : 1];
            {  // U: the rows of plane k along x
                T fv[M], fd[M], r[M];
                load_tab(0, fv, fd);
#pragma unroll
                for (int b = 0; b < M; ++b) {
                    T a0 = 0, a1 = 0, ak = 0;
                    r[b] = ub[i_el + b * BX];
#pragma unroll
                    for (int a = 0; a < M; ++a) {
                        const T v = a == 0 ? r[b] : ub[i_el + b * BX + a];
                        if (!REL || a > 0) {
                            a0 += fv[a] * (REL ? v - r[b] : v);
                            a1 += fd[a] * (REL ? v - r[b] : v);
                        }
                        if constexpr (KF) ak += fv[a] * ub[i_el + NL * 64 + b * BX + a];
                    }
                    A0[b] = a0;
                    A1[b] = a1;
                    if constexpr (KF) AK[b] = ak;
                }
                if constexpr (REL) {
                    w0[kk] = r[0];
#pragma unroll
                    for (int b = 1; b < M; ++b) A0[b] = (A0[b] - A0[0]) + (r[b] - r[0]);
                }
            }
            const T* yt = ytab;
            asm volatile("" : "+s"(yt));  // the y tables are re-read per plane, not kept
#pragma unroll
            for (int y = 0; y < M; ++y) {  // Y
                T s00 = REL ? A0[0] : T(0), s01 = 0, s10 = 0, sk = 0;
#pragma unroll
                for (int b = 0; b < M; ++b) {
                    const T bv = uniform_load(yt + y * 4 * M + b), bd = uniform_load(yt + (y * 4 + 1) * M + b);
                    if (!REL || b > 0) {
                        s00 += bv * A0[b];
                        s01 += bd * A0[b];
                    }
                    s10 += bv * A1[b];
                    if constexpr (KF) sk += bv * AK[b];
                }
                w00[kk][y] = s00;
                w01[kk][y] = s01;
                w10[kk][y] = s10;
                if constexpr (KF) wk[kk][y] = sk;
            }
            // Z of element e, and between its points S of plane e - 1, row by row: the x sums
            // over the Gauss points of an element, entry a = q
            auto points = [&](auto zstage) {
                const T* zt = A.tab[2] + static_cast<long>(ez0 + e) * TAB;
                T tv[M], td[M];
                // (FP32: the z points of a y point together, their sums then added in FP64)
                T dz[M], l0[M], lx[M], ly[M];
#pragma unroll
                for (int p = 0; p < M * M; ++p) {
                    const int z = REL ? p % M : p / M, y = REL ? p / M : p % M, b = p / M;
                    T v[M], vx[M];
                    if (p % M == 0) {
                        if (b == 0) load_tab(2, tv, td);
#pragma unroll
                        for (int r = 0; r < M; ++r) {
                            v[r] = kb[i_k + b * 64 + r];
                            vx[r] = kb[i_k + (M + b) * 64 + r];
                        }
                    }
                    if constexpr (decltype(zstage)::value) {
                        T zv[M], zd[M], zbv[M], zbd[M];
#pragma unroll
                        for (int c = 0; c < M; ++c) {
                            zv[c] = uniform_load(zt + (z * 4 + 0) * M + c);
                            zd[c] = uniform_load(zt + (z * 4 + 1) * M + c);
                            zbv[c] = uniform_load(zt + (z * 4 + 2) * M + c);
                            zbd[c] = uniform_load(zt + (z * 4 + 3) * M + c);
                        }
                        if (REL && z == 0) {  // dz[c]: plane c relative to the first one
                            const int s0 = (kk + 1) % M;
                            dz[0] = w00[s0][y] + w0[REL ? s0 : 0];
#pragma unroll
                            for (int c = 1; c < M; ++c) {
                                const int s = (kk + 1 + c) % M;
                                dz[c] = (w00[s][y] - w00[s0][y]) + (w0[REL ? s : 0] - w0[REL ? s0 : 0]);
                            }
                        }
                        T u = REL ? dz[0] : T(0), ux = 0, uy = 0, uz = 0, kv = 0;
#pragma unroll
                        for (int c = 0; c < M; ++c) {
                            const int s = (kk + 1 + c) % M;
                            if (!REL || c > 0) {
                                if constexpr (MS) u += zv[c] * (REL ? dz[c] : w00[s][y]);
                                uz += zd[c] * (REL ? dz[c] : w00[s][y]);
                            }
                            uy += zv[c] * w01[s][y];
                            ux += zv[c] * w10[s][y];
                            if constexpr (KF) kv += zv[c] * wk[KF ? s : 0][KF ? y : 0];
                        }
                        T g0 = MS ? A.mass * u : T(0);
                        if constexpr (RX) g0 += A.rdt * u * (T(1) - u);
                        // -dt*grad_x is in the x tables, -dt*grad_y and (without a mass term, when
                        // h0 holds u_z alone) -dt*grad_z are applied in T
                        T gx = ux, gy = uy, gz = MS ? A.cz * uz : uz;
                        if constexpr (KF) {
                            gx *= kv;
                            gy *= kv;
                            gz *= kv;
                        }
#pragma unroll
                        for (int c = 0; c < M; ++c) {
                            const int s = (kk + 1 + c) % M;
                            if constexpr (REL) {
                                l0[c] = z == 0 ? zbd[c] * gz : l0[c] + zbd[c] * gz;
                                lx[c] = z == 0 ? zbv[c] * gx : lx[c] + zbv[c] * gx;
                                ly[c] = z == 0 ? zbv[c] * gy : ly[c] + zbv[c] * gy;
                                if constexpr (MS) l0[c] += zbv[c] * g0;
                                if (z == P) {
                                    h0[s][y] = c == P ? l0[c] : h0[s][y] + l0[c];
                                    hx[s][y] = c == P ? lx[c] : hx[s][y] + lx[c];
                                    hy[s][y] = c == P ? ly[c] : hy[s][y] + ly[c];
                                }
                                continue;
                            }
                            if (c == P && z == 0) {  // the element's last plane: its first contribution
                                h0[s][y] = zbd[c] * gz;
                                hx[s][y] = zbv[c] * gx;
                                hy[s][y] = zbv[c] * gy;
                            } else {
                                h0[s][y] += zbd[c] * gz;
                                hx[s][y] += zbv[c] * gx;
                                hy[s][y] += zbv[c] * gy;
                            }
                            if constexpr (MS) h0[s][y] += zbv[c] * g0;
                        }
                    }
                    if (p % M == 0) {
                        T s = 0;
#pragma unroll
                        for (int r = 0; r < M; ++r) {
                            s += tv[r] * v[r];
                            s += td[r] * vx[r];
                        }
                        sb[i_sw + b * M * SX] = el < TX ? s : T(0);
                    }
                }
            };
            if (e >= 0 && e < nzl)
                points(std::true_type{});
            else
                points(std::false_type{});
            wave_lds_sync();
            // plane e - 1 of the wave's rows: one value per DOF (summed in FP64 in both precisions)
#pragma unroll
            for (int j = 0; j < NL; ++j) {
                double v = 0;
#pragma unroll
                for (int a = 0; a < M; ++a) v += static_cast<double>(sb[i_sr[j] + a * (SX - 1)]);
                part[i_pw[j] + (par * M + kk) * L::PLANE] = v;
            }
            {  // T: plane e is complete
                const int s = (kk + 1) % M;
                asm volatile("" : "+s"(yt));
#pragma unroll
                for (int b = 0; b < M; ++b) {
                    T K0 = 0, Ky = 0, Kx = 0;
#pragma unroll
                    for (int y = 0; y < M; ++y) {
                        const T bv = uniform_load(yt + (y * 4 + 2) * M + b), bd = uniform_load(yt + (y * 4 + 3) * M + b);
                        K0 += bv * static_cast<T>(h0[s][y]);
                        Ky += bd * static_cast<T>(hy[s][y]);
                        Kx += bv * static_cast<T>(hx[s][y]);
                    }
                    kb[b * 64 + i_lane] = MS ? K0 + A.cy * Ky : A.cz * K0 + A.cy * Ky;
                    kb[(M + b) * 64 + i_lane] = Kx;
                }
            }
            stage();  // plane k + 1
            fetch(k + 2);
        }
        __syncthreads();  // the planes' sums of all waves are in the part buffer
        write_block(par, k0 - P - 1);
    }
}

template <int P>
double march_tiles(int waves, const int el[3], int tile[3]) {  // its cost, in planes (rhs3_march_pays)
    tile[0] = march<P>::TX;
    tile[1] = kMarchRows;
    // elements per workgroup along z. A workgroup's cost is its elements plus about 2P for the
    // planes without an element at its ends and its start; `cap` workgroups run at once (the waves
    // that march_waves asks for; p = 1 and FP32 up to p = 2 fit 4 to 8 per compute unit), and the
    // last ones to start leave half a round partly idle. Fewer than 4 elements lost everywhere.
    const long columns = static_cast<long>((el[0] + tile[0] - 1) / tile[0]) * ((el[1] + tile[1] - 1) / tile[1]);
    const double cap = 256.0 * waves;
    double best = 0;
    tile[2] = 4;
    for (int nz = 1; nz <= (el[2] + 3) / 4; ++nz) {
        const int tz = std::max(4, (el[2] + nz - 1) / nz);
        const double cost = (tz + 2 * P) * std::max(1.0, columns * ((el[2] + tz - 1) / tz) / cap + 0.5);
        if (nz == 1 || cost < best) {
            best = cost;
            tile[2] = tz;
        }
    }
    return best;
}

}  // namespace

double rhs3_march_tiles(int p, int bytes, bool kfield, const int elements[3], int tile[3], int nt[3]) {
    const int waves = march_waves(bytes, p, kfield);
    const double cost = p == 1   ? march_tiles<1>(waves, elements, tile)
                        : p == 2 ? march_tiles<2>(waves, elements, tile)
                                 : march_tiles<3>(waves, elements, tile);
    for (int d = 0; d < 3; ++d) nt[d] = (elements[d] + tile[d] - 1) / tile[d];
    return cost;
}

namespace {

template <typename T, int P, bool KF, int FM>
hipError_t march_launch(const T* up, T* rhs, const dev_tables<T>* d, const rhs_params<T>& prm, const int tile[3],
                        const int nt[3], hipStream_t s) {
    const long blocks = static_cast<long>(nt[0]) * nt[1] * nt[2];
    if (tile[0] != march<P>::TX || tile[1] != kMarchRows || tile[2] < P ||
        !rhs3_march_fits(sizeof(T), d[0].dofs, d[1].dofs, nt))
        return hipErrorInvalidValue;
    march_args<T> a;
    a.up = up;
    a.kfield = prm.kfield;
    a.rhs = rhs;
    a.start = prm.start ? prm.start : prm.store ? nullptr : rhs;
    a.scale = prm.start ? prm.start_scale : T(1);
    a.spill = prm.spill;
    for (int i = 0; i < 3; ++i) {
        a.tab[i] = d[i].pack;
        a.n[i] = d[i].dofs;
        a.el[i] = d[i].elements;
        a.ext[i][0] = prm.spill_ext[i][0];
        a.ext[i][1] = prm.spill_ext[i][1];
        if (!a.tab[i]) return hipErrorInvalidValue;
    }
    for (int k = 0; k < 8; ++k) a.off[k] = prm.spill_off[k];
    a.ntx = nt[0];
    a.nty = nt[1];
    a.tz = tile[2];
    a.cx = -prm.dt * prm.gx;
    a.cy = -prm.dt * prm.gy;
    a.cz = -prm.dt * prm.gz;
    a.mass = prm.mass;
    a.rdt = prm.dt * prm.reaction;
    auto kern = k_rhs3_march<T, P, KF, FM>;
    constexpr size_t shm = march_lds<T, P, KF>::bytes();
    static_assert(shm <= 160 * 1024, "the workgroup's LDS");
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                              static_cast<int>(shm));
    hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(blocks)), dim3(64 * kMarchRows), shm, s, a);
    return hipGetLastError();
}

template <typename T, int P>
hipError_t march_forms(const T* up, T* rhs, const dev_tables<T>* d, const rhs_params<T>& prm, const int tile[3],
                       const int nt[3], hipStream_t s) {
    const bool rx = prm.reaction != T(0), ms = rx || prm.mass != T(0);
    if constexpr (!rhs3_march_kfield<T>(P)) {
        if (prm.kfield) return hipErrorInvalidValue;
    } else if (prm.kfield) {
        if (rx) return march_launch<T, P, true, 1>(up, rhs, d, prm, tile, nt, s);
        return ms ? march_launch<T, P, true, 0>(up, rhs, d, prm, tile, nt, s)
                  : march_launch<T, P, true, 2>(up, rhs, d, prm, tile, nt, s);
    }
    if (rx) return march_launch<T, P, false, 1>(up, rhs, d, prm, tile, nt, s);
    return ms ? march_launch<T, P, false, 0>(up, rhs, d, prm, tile, nt, s)
              : march_launch<T, P, false, 2>(up, rhs, d, prm, tile, nt, s);
}

}  // namespace

template <typename T>
hipError_t launch_rhs3_march(int p, const T* u_prev, T* rhs, const dev_tables<T>* dirs, const rhs_params<T>& prm,
                             const int tile[3], const int nt[3], hipStream_t s) {
    if (!prm.spill) return hipErrorInvalidValue;
    switch (p) {
        case 1:
            return march_forms<T, 1>(u_prev, rhs, dirs, prm, tile, nt, s);
        case 2:
            return march_forms<T, 2>(u_prev, rhs, dirs, prm, tile, nt, s);
        case 3:
            return march_forms<T, 3>(u_prev, rhs, dirs, prm, tile, nt, s);
        default:
            return hipErrorInvalidValue;
    }
}

template hipError_t launch_rhs3_march<double>(int, const double*, double*, const dev_tables<double>*,
                                              const rhs_params<double>&, const int*, const int*, hipStream_t);
template hipError_t launch_rhs3_march<float>(int, const float*, float*, const dev_tables<float>*,
                                             const rhs_params<float>&, const int*, const int*, hipStream_t);

}  // namespace adsg

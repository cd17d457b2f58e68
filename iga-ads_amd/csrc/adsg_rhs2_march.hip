// HIP element-loop RHS of the MI355X ADS step in 2D (gfx950) in one launch without spill
// entries: the integrals of compute_rhs (validation.hpp:95-119) for one problem or for a
// batch of problems of every degree.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "adsg_device.hpp"

namespace adsg {

namespace {

// ------------------------------------------------------------------------------------
// Sum factorisation shared by the elements of a column. A wave owns a strip of 64 - P DOF
// columns and A.rows DOF rows; lane l is element column e = e0 + l, e0 = (first column) - P,
// and it also owns DOF column e. The wave marches along y. Per DOF row:
//  X  its M = P + 1 coefficients of the row contracted along x at its M Gauss points (value,
//     derivative), kept in registers for the M rows that an element row reads,
//  Y  for the element row that begins at this DOF row: along y to the M^2 Gauss points, the
//     integrand, and its y-transposed sums (FP32: transposed in x too), kept in FP64 registers
//     for the M rows it touches,
//  S  the row is complete: x transposed (FP64), the M contributions to neighbouring columns summed
//     by shifting them across the lanes, stored.
// The x contractions run once per DOF row instead of once per element, and every DOF is
// written once by one lane in a fixed order: no colours, no spill entries, no LDS. What it
// costs is P of 64 lanes and P element rows per strip computed twice.
// Bound: instruction issue, and in small problems the serial P + 1 element rows of a strip.
// Whole steps, us, element kernel in 16 x 16 tiles (four colour launches in batches, one launch
// and a spill fix-up for one problem) and here: 256 problems of 32 to 256 elements FP32 289 ->
// 191 (of them the element kernels 186 -> 96), 24 of 32 to 90 110 -> 36, 96 of 32 to 200 FP64
// 155 -> 103 (sweeps and all). One problem, FP64, element kernel and fix-up: 128 x 128 p = 2
// with a k field 8.3 -> 5.6, 480 x 351 p = 3 25 -> 17.
// ------------------------------------------------------------------------------------

// lane l: the value of lane l - 1, 0 in lane 0 (DPP wave_shr:1)
__device__ __forceinline__ int lane_below(int v) { return __builtin_amdgcn_update_dpp(0, v, 0x138, 0xf, 0xf, false); }
__device__ __forceinline__ double lane_below(double v) {
    return __hiloint2double(lane_below(__double2hiint(v)), lane_below(__double2loint(v)));
}

__device__ __forceinline__ float mad(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double mad(double a, double b, double c) { return __builtin_fma(a, b, c); }

// (every multiply-add is written out, so that the kernels this is part of round alike: a problem
// of a batch equals the problem run alone bit for bit)
template <typename T, int P, bool KF>
__device__ __forceinline__ void march2_strip(const march2_args<T>& A, int t) {
#pragma clang fp contract(off)
    constexpr int M = P + 1;
    const int lane = threadIdx.x & 63;
    const int tx = t % A.ntx, ty = t / A.ntx;
    const int e = tx * (64 - P) - P + lane;
    const bool in = e >= 0 && e < A.ex;
    const int ec = min(max(e, 0), A.ex - 1);
    const int r0 = ty * A.rows, r1 = min(r0 + A.rows, A.ny), b0 = max(r0 - P, 0);

    // x tables of the lane's element: values, derivatives and weights at its Gauss points
    T bv[M][M], bd[M][M], wx[M];
#pragma unroll
    for (int q = 0; q < M; ++q) {
#pragma unroll
        for (int i = 0; i < M; ++i) {
            bv[q][i] = A.xv[(ec * M + q) * M + i];
            bd[q][i] = A.xd[(ec * M + q) * M + i];
        }
        wx[q] = A.xw[ec * M + q];
    }
    const T* up = A.up + ec;
    const T* kp = KF ? A.kfield + ec : nullptr;
    T nu[M], nk[KF ? M : 1];  // the next DOF row, on its way
    auto fetch = [&](int r) {
        const long o = static_cast<long>(A.nx) * min(r, A.ny - 1);
#pragma unroll
        for (int i = 0; i < M; ++i) {
            nu[i] = up[o + i];
            if constexpr (KF) nk[i] = kp[o + i];
        }
    };
    // Values are kept relative to the row's first coefficient and summed from differences, which
    // the derivatives are made of: their rounding errors scale with the differences, not with u
    // (the basis functions sum to 1 and their derivatives to 0).
    T a[M][M], d[M][M], u0[M], k[KF ? M : 1][KF ? M : 1];  // [DOF row][x Gauss point]
    auto contract = [&](int j) {
        u0[j] = nu[0];
#pragma unroll
        for (int i = 1; i < M; ++i) nu[i] -= nu[0];
#pragma unroll
        for (int q = 0; q < M; ++q) {
            T s = 0, sd = 0, sk = 0;
#pragma unroll
            for (int i = 0; i < M; ++i) {
                if (i > 0) s = mad(bv[q][i], nu[i], s);
                if (i > 0) sd = mad(bd[q][i], nu[i], sd);
                if constexpr (KF) sk = mad(bv[q][i], nk[i], sk);
            }
            a[j][q] = s;
            d[j][q] = sd;
            if constexpr (KF) k[j][q] = sk;
        }
    };
    // The sums of row r + j. The sums of different elements are FP64 in both precisions. FP64:
    // against values (V) and x derivatives (D) at the lane's Gauss points, x transposed once per
    // row. FP32: an element's contributions are complete in FP32 before they are added, R[j][i] to
    // its column i: sums across element rows first and x transposed after them in FP32 were 10 to
    // 20 % further from FP64 on rough states (and tables with the weights folded in up to 30 % at
    // p = 1: their rounding is the same in every element).
    constexpr bool F32 = sizeof(T) == sizeof(float);
    constexpr int MV = F32 ? 1 : M, MR = F32 ? M : 1;
    double V[MV][MV], D[MV][MV], R[MR][MR];
    const T cx = A.cx;
#pragma unroll
    for (int j = 0; j < MV; ++j)
#pragma unroll
        for (int q = 0; q < MV; ++q) V[j][q] = D[j][q] = 0.0;
#pragma unroll
    for (int j = 0; j < MR; ++j)
#pragma unroll
        for (int i = 0; i < MR; ++i) R[j][i] = 0.0;
    fetch(b0);
#pragma unroll
    for (int j = 0; j < P; ++j) {
        contract(j);
        fetch(b0 + j + 1);
    }

    const T* start = A.start ? A.start + e : nullptr;
    T* out = A.rhs + e;
    const bool own = lane >= P && e < A.nx;
    for (int r = b0; r < r1; ++r) {
        if (r < A.ey) {
            contract(P);
            fetch(r + M);
            const T *yv = A.yv + r * M * M, *yd = A.yd + r * M * M, *yw = A.yw + r * M;
            // the value term: 0 none, 1 the mass term, 2 with the reaction
            auto element = [&](auto value_term) {
                constexpr int VAL = decltype(value_term)::value;
                T da[M][M];  // rows relative to the first one
#pragma unroll
                for (int q = 0; q < M; ++q) {
                    da[0][q] = a[0][q] + u0[0];
#pragma unroll
                    for (int c = 1; c < M; ++c) da[c][q] = (a[c][q] - a[0][q]) + (u0[c] - u0[0]);
                }
                T lv[M], ld[M], sum[MR][MR];  // FP32: the y points of an x point, its sums; the element's
#pragma unroll
                for (int o = 0; o < M; ++o) {
#pragma unroll
                    for (int i = 0; i < M; ++i) {
                        const int y = F32 ? i : o, q = F32 ? o : i;
                        T v[M], g[M];
#pragma unroll
                        for (int c = 0; c < M; ++c) {
                            v[c] = (uniform_load(yv + y * M + c));
                            g[c] = (uniform_load(yd + y * M + c));
                        }
                        const T w = (uniform_load(yw + y)), wc = w * A.cy;
                        const T wm = VAL == 2 ? w * (A.mass + A.rdt) : w * A.mass, wr = w * A.rdt;
                        T u = da[0][q], ux = 0, uy = 0, kv = 0;
#pragma unroll
                        for (int c = 0; c < M; ++c) {
                            if (c > 0) {
                                if constexpr (VAL > 0) u = mad(v[c], da[c][q], u);
                                uy = mad(g[c], da[c][q], uy);
                            }
                            ux = mad(v[c], d[c][q], ux);
                            if constexpr (KF) kv = mad(v[c], k[c][q], kv);
                        }
                        T gx = w * ux, gy = wc * uy;
                        if constexpr (KF) {
                            gx *= kv;
                            gy *= kv;
                        }
                        u *= VAL == 2 ? mad(-wr, u, wm) : wm;  // w (mass u + dt reaction u (1 - u))
#pragma unroll
                        for (int c = 0; c < M; ++c) {
                            if constexpr (F32) {
                                lv[c] = y == 0 ? g[c] * gy : mad(g[c], gy, lv[c]);
                                if constexpr (VAL > 0) lv[c] = mad(v[c], u, lv[c]);
                                ld[c] = y == 0 ? v[c] * gx : mad(v[c], gx, ld[c]);
                                if (y == P) {
                                    lv[c] *= wx[q];
                                    ld[c] *= cx * wx[q];
#pragma unroll
                                    for (int x = 0; x < M; ++x) {
                                        sum[c][x] = q == 0 ? bv[q][x] * lv[c] : mad(bv[q][x], lv[c], sum[c][x]);
                                        sum[c][x] = mad(bd[q][x], ld[c], sum[c][x]);
                                        if (q == P) R[c][x] += sum[c][x];
                                    }
                                }
                            } else {
                                V[c][q] = mad(g[c], gy, V[c][q]);
                                if constexpr (VAL > 0) V[c][q] = mad(v[c], u, V[c][q]);
                                D[c][q] = mad(v[c], gx, D[c][q]);
                            }
                        }
                    }
                }
            };
            if (A.rdt != T(0))
                element(std::integral_constant<int, 2>{});
            else if (A.mass != T(0))
                element(std::integral_constant<int, 1>{});
            else
                element(std::integral_constant<int, 0>{});
        }
        // row r is complete
        double s = 0;
#pragma unroll
        for (int i = P; i >= 0; --i) {
            double c = 0;
            if constexpr (F32) {
                c = R[0][i];
            } else {
#pragma unroll
                for (int q = 0; q < M; ++q) {
                    c = mad(bv[q][i], wx[q] * V[0][q], c);
                    c = mad(bd[q][i], (cx * wx[q]) * D[0][q], c);
                }
            }
            s = (i < P ? lane_below(s) : 0.0) + (in ? c : 0.0);
        }
        if (r >= r0 && own) {
            const long o = static_cast<long>(A.nx) * r;
            out[o] = start ? mad(A.scale, start[o], static_cast<T>(s)) : static_cast<T>(s);
        }
#pragma unroll
        for (int j = 0; j < P; ++j) {
            u0[j] = u0[j + 1];
#pragma unroll
            for (int q = 0; q < M; ++q) {
                a[j][q] = a[j + 1][q];
                d[j][q] = d[j + 1][q];
                if constexpr (KF) k[j][q] = k[j + 1][q];
                if constexpr (F32) {
                    R[j][q] = R[j + 1][q];
                } else {
                    V[j][q] = V[j + 1][q];
                    D[j][q] = D[j + 1][q];
                }
            }
        }
#pragma unroll
        for (int q = 0; q < M; ++q) {
            if constexpr (F32)
                R[P][q] = 0.0;
            else
                V[P][q] = D[P][q] = 0.0;
        }
    }
}

// waves per SIMD the register allocation must allow: the windows, the sums and the x tables
// are 6 M^2 values per lane (7 M^2 with a k field)
template <typename T, int P, bool KF>
constexpr int march2_waves() {
    return sizeof(T) == sizeof(float) ? (P == 3 && KF ? 2 : 3) : P == 3 ? 1 : 2;
}

template <typename T, int P, bool KF>
__global__ __launch_bounds__(64, (march2_waves<T, P, KF>())) void k_rhs2_march(march2_args<T> A) {
    march2_strip<T, P, KF>(A, xcd_contiguous(blockIdx.x, gridDim.x));
}

// Every degree in one launch, the highest first: the strips of p = 3 take longest and those of
// p = 1 fill the chip while the last of them end (three launches, one per degree: 121 us
// against 95 for 256 problems of 32 to 256 elements in FP32).
template <typename T>
__global__ __launch_bounds__(64, (sizeof(T) == sizeof(float) ? 3 : 2)) void k_rhs2_march_batch(
    const march2_item<T>* __restrict__ items, int nitems) {
    const int b = blockIdx.x;
    int lo = 0, hi = nitems - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) / 2;
        if (items[mid].first <= b)
            lo = mid;
        else
            hi = mid - 1;
    }
    const march2_item<T>& it = items[lo];
    const int p = it.p;  // uniform
    if (p == 3) march2_strip<T, 3, false>(it.a, b - it.first);
    if (p == 2) march2_strip<T, 2, false>(it.a, b - it.first);
    if (p == 1) march2_strip<T, 1, false>(it.a, b - it.first);
}

template <typename T, int P>
hipError_t march2_launch(const march2_args<T>& a, unsigned blocks, hipStream_t s) {
    if (a.kfield)
        hipLaunchKernelGGL((k_rhs2_march<T, P, true>), dim3(blocks), dim3(64), 0, s, a);
    else
        hipLaunchKernelGGL((k_rhs2_march<T, P, false>), dim3(blocks), dim3(64), 0, s, a);
    return hipGetLastError();
}

}  // namespace

int march2_rows(int bytes, const std::vector<std::array<int, 3>>& problems) {
    // DOF rows per strip. A strip costs its rows and about p + 3 more (the element rows it
    // shares, its first rows' contractions, its tables), a row of p = 1, 2, 3 about 0.2, 0.45,
    // 1 of a p = 3 row. One FP64 wave, or two FP32 waves, fill a SIMD. One problem: rounds of
    // whole strips, one per SIMD (p = 3 FP64 480 x 351 us: 2 rows 24.5, 3 17.0, 4 17.7, 6 20.0);
    // a batch: the mean load and the longest strip (256 problems of 32 to 256 elements FP32, us
    // per step: 4 rows 210, 8 191, 16 183, 32 194; 96 of 32 to 200 FP64: 4 116, 6 100, 12 106).
    static const int kRows[] = {1, 2, 3, 4, 5, 6, 8, 10, 12, 16, 20, 24, 32, 40, 48, 64, 96, 128};
    static const double kWeight[4] = {0, 0.2, 0.45, 1};
    const double cap = bytes == 4 ? 2048 : 1024;
    int best = 1;
    double least = 0;
    for (int rows : kRows) {
        double load = 0, longest = 0;
        for (const auto& q : problems) {
            const int p = q[0], cols = 64 - p;
            const double n = static_cast<double>((q[1] + cols - 1) / cols) * ((q[2] + rows - 1) / rows);
            const double t = kWeight[p] * (rows + p + 3.0);
            load += n * t / cap;
            longest = std::max(longest, t);
        }
        const double cost = problems.size() == 1 ? longest * std::ceil(load / longest) : load + longest;
        if (least == 0 || cost < least) {
            least = cost;
            best = rows;
        }
    }
    return best;
}

template <typename T>
march2_args<T> march2_problem(int p, int rows, const T* up, T* rhs, const dev_tables<T>& X, const dev_tables<T>& Y,
                              const rhs_params<T>& prm) {
    march2_args<T> a;
    a.up = up;
    a.kfield = prm.kfield;
    a.start = prm.start ? prm.start : prm.store ? nullptr : rhs;
    a.scale = prm.start ? prm.start_scale : T(1);
    a.rhs = rhs;
    a.xv = X.val;
    a.xd = X.der;
    a.xw = X.wj;
    a.yv = Y.val;
    a.yd = Y.der;
    a.yw = Y.wj;
    a.nx = X.dofs;
    a.ny = Y.dofs;
    a.ex = X.elements;
    a.ey = Y.elements;
    a.ntx = (a.nx + 63 - p) / (64 - p);
    a.rows = rows;
    a.mass = prm.mass;
    a.rdt = prm.dt * prm.reaction;
    a.cx = -prm.dt * prm.gx;
    a.cy = -prm.dt * prm.gy;
    return a;
}

template <typename T>
hipError_t launch_rhs2_march(int p, const T* up, T* rhs, const dev_tables<T>* d, const rhs_params<T>& prm,
                             hipStream_t s) {
    if (d[0].dofs != d[0].elements + p || d[1].dofs != d[1].elements + p) return hipErrorInvalidValue;
    const int rows = march2_rows(sizeof(T), {{p, d[0].dofs, d[1].dofs}});
    const march2_args<T> a = march2_problem<T>(p, rows, up, rhs, d[0], d[1], prm);
    const unsigned blocks = static_cast<unsigned>(march2_strips(a));
    if (p == 1) return march2_launch<T, 1>(a, blocks, s);
    if (p == 2) return march2_launch<T, 2>(a, blocks, s);
    if (p == 3) return march2_launch<T, 3>(a, blocks, s);
    return hipErrorInvalidValue;
}

template <typename T>
hipError_t launch_rhs2_march_batch(const march2_item<T>* items, int nitems, int blocks, hipStream_t s) {
    if (blocks <= 0 || nitems <= 0) return hipSuccess;
    hipLaunchKernelGGL((k_rhs2_march_batch<T>), dim3(blocks), dim3(64), 0, s, items, nitems);
    return hipGetLastError();
}

#define ADSG_INST(T)                                                                                               \
    template march2_args<T> march2_problem<T>(int, int, const T*, T*, const dev_tables<T>&, const dev_tables<T>&,   \
                                              const rhs_params<T>&);                                               \
    template hipError_t launch_rhs2_march<T>(int, const T*, T*, const dev_tables<T>*, const rhs_params<T>&,         \
                                             hipStream_t);                                                         \
    template hipError_t launch_rhs2_march_batch<T>(const march2_item<T>*, int, int, hipStream_t);
ADSG_INST(double)
ADSG_INST(float)
#undef ADSG_INST

}  // namespace adsg

// HIP element-loop RHS of the MI355X ADS step (gfx950): compute_rhs (validation.hpp:95-119)
// with one workgroup per tile of elements, one lane per element, sum factorisation through
// the 1D tables, local contributions combined in LDS, and tiles of one parity colour
// (2^d colours) adding their DOF blocks into the global rhs without atomics. The tiles can
// also run in one launch: each tile adds the block entries it owns and spills the rest,
// which a second kernel (k_rhs_fixup; in a step, at the start of the sweep phase) adds in a
// fixed order (deterministic either way). The adjoint's k-field gradient runs on the same
// tiles.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "adsg_device.hpp"
#include "adsg_kernels.hpp"

namespace adsg {

namespace {

// ------------------------------------------------------------------------------------
// element-loop RHS, 3D
// ------------------------------------------------------------------------------------
// VAR 0: hold the element's coefficient block in registers (fewer LDS reads); 1: re-read it
// from LDS for every x Gauss point (fewer registers: two waves per SIMD); 2: as 1, and the
// element's contribution is added to the LDS planes after every x Gauss point instead of
// being accumulated in registers (fewer registers again; FP32 runs four waves per SIMD);
// 3: two tiles per workgroup, the second copied global-to-LDS while the first is integrated
// (k_rhs3_pipe); 4: each wave integrates two element layers and carries their shared DOF
// planes in registers (k_rhs3_zpair, p <= 2).
//
// One lane per element; the x/y tables of the tile's elements are staged in LDS, the
// forward ones as tabulated and the backward ones with the quadrature weight (and, for the
// derivative tables, the constant -dt*grad_d) folded in, so that the only per-point work
// is the integrand itself. The element contributions are summed per wave into private DOF
// planes with LDS atomic adds: a wave's adds are executed in instruction order, so the sums
// are deterministic, and waves never share a plane. One barrier later the planes of the
// (P+1) waves that touch a DOF plane are added and the tile's block is added into the rhs.
template <typename T, int P, int VAR>
constexpr int rhs3_waves() {  // minimum waves per SIMD the register allocation must allow
    return VAR == 0 ? 1 : VAR == 1 || VAR == 3 || VAR == 4 ? 2 : P == 3 ? 2 : sizeof(T) == sizeof(float) ? 4 : 3;
}

// first element of tile t of the given parity colour (ntx2, nty2 tiles of that colour per
// tile row and tile plane)
struct tile3 {
    int ex0, ey0, ez0;
};
template <int TX, int TY, int TZ>
__device__ __forceinline__ tile3 rhs3_tile(int t, int colour, int ntx2, int nty2) {
    const int tx = 2 * (t % ntx2) + (colour & 1);
    t /= ntx2;
    const int ty = 2 * (t % nty2) + ((colour >> 1) & 1);
    t /= nty2;
    const int tz = 2 * t + ((colour >> 2) & 1);
    return {tx * TX, ty * TY, tz * TZ};
}
// tile t of the launch: of the given colour, or (ONE) of all ntx x nty x ntz tiles
template <bool ONE, int TX, int TY, int TZ>
__device__ __forceinline__ tile3 rhs3_tile_of(int t, int colour, int ntx, int nty) {
    if constexpr (ONE) {
        const int tx = t % ntx;
        t /= ntx;
        return {tx * TX, (t % nty) * TY, (t / nty) * TZ};
    } else {
        return rhs3_tile<TX, TY, TZ>(t, colour, ntx, nty);
    }
}

// Where a tile's block sums go. Colour launches (ONE false): every entry is added to the
// rhs with a return-less global add; the tiles of one colour share no DOF, so each DOF has
// one writer per launch. One launch over all tiles (ONE true): tile t owns DOF index g of a
// direction when t T <= g < (t + 1) T, or t T <= g in the direction's last tile, so every
// DOF has one owner; the owner adds its entry to the rhs (a plain read-modify-write: no
// other workgroup writes it; a store when the rhs start value is unused) and the other tiles
// store theirs in the spill arrays, which k_rhs_fixup adds to the rhs afterwards in a fixed
// order. An entry whose owner lies at offset delta from the tile (delta_d = 1 where the
// entry is in the tile's top P layers of direction d and the tile is not the last there)
// goes to array delta at the DOF's own index in the directions with delta_d = 0 and at
// t_d P + l_d (owner tile t_d, local index l_d < P) in the others: the fix-up then reads
// every array at consecutive addresses for consecutive DOFs.
template <typename T>
struct block_sink {
    T* rhs;
    int tile[3];   // ONE: the tile's indices
    bool last[3];  // ONE: the tile is the last of its direction
};
template <bool ONE, int TX, int TY, int TZ, typename T>
__device__ __forceinline__ block_sink<T> rhs3_sink(T* rhs, tile3 o, int ex, int ey, int ez) {
    if constexpr (ONE)
        return {rhs, {o.ex0 / TX, o.ey0 / TY, o.ez0 / TZ}, {o.ex0 + TX >= ex, o.ey0 + TY >= ey, o.ez0 + TZ >= ez}};
    else
        return {rhs, {0, 0, 0}, {false, false, false}};
}
// entry (bx, by, bz) of the block, DOF (gx, gy, gz) = g of the mesh
template <bool ONE, int P, int TX, int TY, int TZ, typename T>
__device__ __forceinline__ void rhs3_put(const block_sink<T>& k, const rhs_params<T>& prm, int bx, int by, int bz,
                                         int gx, int gy, int gz, long g, double sum) {
    if constexpr (ONE) {
        const int dx = bx >= TX && !k.last[0], dy = by >= TY && !k.last[1], dz = bz >= TZ && !k.last[2];
        if (!(dx | dy | dz)) {
            k.rhs[g] = prm.store ? static_cast<T>(sum) : k.rhs[g] + static_cast<T>(sum);
        } else {
            const int cx = dx ? (k.tile[0] + 1) * P + bx - TX : gx;
            const int cy = dy ? (k.tile[1] + 1) * P + by - TY : gy;
            const int cz = dz ? (k.tile[2] + 1) * P + bz - TZ : gz;
            prm.spill[spill_index(prm, dx, dy, dz, cx, cy, cz)] = static_cast<T>(sum);
        }
    } else {
        unsafeAtomicAdd(k.rhs + g, static_cast<T>(sum));
    }
}

// The LDS data of one tile: its coefficient block (and k / f blocks) and the x and y tables
// of its elements: xt[FV], xt[FD] as tabulated, xt[BV], xt[BD] with the quadrature weight
// (variants 0-2 also fold -dt*grad_x into xt[BD], -dt*grad_y into yt[BD]).
enum { FV = 0, FD = 1, BV = 2, BD = 3 };
template <typename T, int P, int TX, int TY, int TZ, bool KF>
struct rhs3_buf {
    static constexpr int M = P + 1, BX = TX + P, BY = TY + P, BZ = TZ + P;
    static constexpr int NB = BX * BY * BZ, PL = BX * BY;
    T blk[NB];
    T kb[KF ? NB : 1];
    T xt[4][TX * M * M];
    T yt[4][TY * M * M];
};
// the waves' private DOF planes (wave lz owns planes lz*M .. lz*M+P, DOF z = lz + c; FP64 in
// both precisions: the FP64 LDS add is the fast one on this part)
template <int P, int TX, int TY, int TZ>
constexpr int rhs3_acc_size() {
    return TZ * (P + 1) * (TX + P) * (TY + P);
}
// The LDS of a workgroup with NBUF tile buffers and their planes, in one object: the
// compiler then addresses every part from one base (separate __shared__ arrays cost
// registers in the element loop).
template <typename T, int P, int TX, int TY, int TZ, bool KF, int NBUF>
struct rhs3_lds {
    rhs3_buf<T, P, TX, TY, TZ, KF> b[NBUF];
    double acc[NBUF][rhs3_acc_size<P, TX, TY, TZ>()];
};

// One element (lane lx, ly of wave lz) of the tile whose first element is (ex0, ey0, ez0):
// sum-factorised integrand over its Gauss points, its contribution accumulated in R (owned
// and zeroed by the caller) and added to the wave's planes, or (variant 4) left in R for
// the caller, which carries the planes shared with the wave's next element layer.
template <typename T, int P, int TX, int TY, int TZ, bool KF, int FM, int VAR>
__device__ __forceinline__ void rhs3_element(const rhs3_buf<T, P, TX, TY, TZ, KF>& L,
                                             double* acc, const dev_tables<T>& X,
                                             const dev_tables<T>& Y, const dev_tables<T>& Z,
                                             const rhs_params<T>& prm, int lx, int ly, int lz,
                                             int ex0, int ey0, int ez0,
                                             T (&R)[P + 1][P + 1][P + 1]) {
    using LDS = rhs3_buf<T, P, TX, TY, TZ, KF>;
    constexpr int M = P + 1, BX = LDS::BX, BY = LDS::BY, PL = LDS::PL;
    constexpr bool CREG = VAR == 0;  // coefficient block held in registers
    // element contribution added to the planes per x point (variant 3 at P = 3: registers)
    constexpr bool FLUSH = VAR == 2 || (VAR == 3 && P == 3);
    constexpr bool TW = VAR == 3;  // tables weighted only: -dt*grad applied as read
    // FM: 0 the heat form (mass term), 1 with the reaction term, 2 no mass term (mass = 0, no
    // reaction: the delta and FP32 increment forms), where u itself is not needed
    constexpr bool RX = FM == 1, MS = FM != 2;
    static_assert(MS || !RX, "form 2 has no term in v other than the gradient terms");
    static_assert(VAR != 4 || P <= 2, "variant 4 carries the register block: p <= 2");
    const int ez = ez0 + lz;
    // the wave's planes: in one add instruction the 64 lanes hit 64 distinct entries
    double* mine = acc + lz * M * PL;


    if (ez < Z.elements) {  // wave-uniform
        // z tables of the wave's element layer: uniform addresses in uniform control flow,
        // read with scalar loads
        T Bz[M][M], Dz[M][M], wz[M];
        const T* zv = Z.val + static_cast<long>(ez) * M * M;
        const T* zd = Z.der + static_cast<long>(ez) * M * M;
#pragma unroll
        for (int q = 0; q < M; ++q) {
            wz[q] = uniform_load(Z.wj + static_cast<long>(ez) * M + q);
#pragma unroll
            for (int c = 0; c < M; ++c) {
                Bz[q][c] = uniform_load(zv + q * M + c);
                Dz[q][c] = uniform_load(zd + q * M + c);
            }
        }
        const T cz = -prm.dt * prm.gz;
        const T cx = -prm.dt * prm.gx, cy = -prm.dt * prm.gy;  // used by TW only
        // per z point constants with the weight folded in (wave-uniform)
        T mwz[M], cwz[M], rwz[M];
#pragma unroll
        for (int q = 0; q < M; ++q) {
            mwz[q] = prm.mass * wz[q];
            cwz[q] = cz * wz[q];
            rwz[q] = prm.dt * prm.reaction * wz[q];
        }
        if (ex0 + lx < X.elements && ey0 + ly < Y.elements) {
            T cf[CREG ? M : 1][CREG ? M : 1][CREG ? M : 1];
            T kc[KF && CREG ? M : 1][KF && CREG ? M : 1][KF && CREG ? M : 1];
            if constexpr (CREG) {
#pragma unroll
                for (int a = 0; a < M; ++a)
#pragma unroll
                    for (int b = 0; b < M; ++b)
#pragma unroll
                        for (int c = 0; c < M; ++c) {
                            const int li = (lx + a) + BX * ((ly + b) + BY * (lz + c));
                            cf[a][b][c] = L.blk[li];
                            if constexpr (KF) kc[a][b][c] = L.kb[li];
                        }
            }
#pragma unroll 1
            for (int qx = 0; qx < M; ++qx) {
                T bx[M], dx[M];
#pragma unroll
                for (int a = 0; a < M; ++a) {
                    bx[a] = L.xt[FV][(lx * M + qx) * M + a];
                    dx[a] = L.xt[FD][(lx * M + qx) * M + a];
                }
                // stage x: contract the element's first index
                T A0[M][M], A1[M][M], KA[KF ? M : 1][KF ? M : 1];
#pragma unroll
                for (int b = 0; b < M; ++b)
#pragma unroll
                    for (int c = 0; c < M; ++c) {
                        T s0 = 0, s1 = 0, sk = 0;
#pragma unroll
                        for (int a = 0; a < M; ++a) {
                            const int li = (lx + a) + BX * ((ly + b) + BY * (lz + c));
                            const T cv = CREG ? cf[CREG ? a : 0][CREG ? b : 0][CREG ? c : 0] : L.blk[li];
                            s0 += bx[a] * cv;
                            s1 += dx[a] * cv;
                            if constexpr (KF)
                                sk += bx[a] * (CREG ? kc[KF && CREG ? a : 0][KF && CREG ? b : 0][KF && CREG ? c : 0] : L.kb[li]);
                        }
                        A0[b][c] = s0;
                        A1[b][c] = s1;
                        if constexpr (KF) KA[b][c] = sk;
                    }
                T K0[M][M], Kx[M][M];
#pragma unroll
                for (int b = 0; b < M; ++b)
#pragma unroll
                    for (int c = 0; c < M; ++c) K0[b][c] = Kx[b][c] = T(0);
#pragma unroll 1
                for (int qy = 0; qy < M; ++qy) {
                    T by[M], dy[M];
#pragma unroll
                    for (int b = 0; b < M; ++b) {
                        by[b] = L.yt[FV][(ly * M + qy) * M + b];
                        dy[b] = L.yt[FD][(ly * M + qy) * M + b];
                    }
                    // stage y for this Gauss point
                    T a00[M], a01[M], a10[M], ka[KF ? M : 1];
#pragma unroll
                    for (int c = 0; c < M; ++c) {
                        T s00 = 0, s01 = 0, s10 = 0, sk = 0;
#pragma unroll
                        for (int b = 0; b < M; ++b) {
                            s00 += by[b] * A0[b][c];
                            s01 += dy[b] * A0[b][c];
                            s10 += by[b] * A1[b][c];
                            if constexpr (KF) sk += by[b] * KA[b][c];
                        }
                        a00[c] = s00;
                        a01[c] = s01;
                        a10[c] = s10;
                        if constexpr (KF) ka[c] = sk;
                    }
                    T H0[M], Hx[M], Hy[M];
#pragma unroll
                    for (int c = 0; c < M; ++c) H0[c] = Hx[c] = Hy[c] = T(0);
#pragma unroll
                    for (int qz = 0; qz < M; ++qz) {
                        // stage z, the integrand, and stage z transposed
                        T u = 0, uz = 0, uy = 0, ux = 0, kv = 0;
#pragma unroll
                        for (int c = 0; c < M; ++c) {
                            if constexpr (MS) u += Bz[qz][c] * a00[c];
                            uz += Dz[qz][c] * a00[c];
                            uy += Bz[qz][c] * a01[c];
                            ux += Bz[qz][c] * a10[c];
                            if constexpr (KF) kv += Bz[qz][c] * ka[c];
                        }
                        T g0 = MS ? mwz[qz] * u : T(0);
                        if constexpr (RX) g0 += rwz[qz] * u * (T(1) - u);
                        T gx, gy, gz;
                        if constexpr (KF) {
                            const T kw = wz[qz] * kv;
                            gx = kw * ux;
                            gy = kw * uy;
                            gz = (cz * kw) * uz;
                        } else {
                            gx = wz[qz] * ux;
                            gy = wz[qz] * uy;
                            gz = cwz[qz] * uz;
                        }
#pragma unroll
                        for (int c = 0; c < M; ++c) {  // separate updates: two FMAs, no add
                            if constexpr (MS) H0[c] += Bz[qz][c] * g0;
                            H0[c] += Dz[qz][c] * gz;
                            Hx[c] += Bz[qz][c] * gx;
                            Hy[c] += Bz[qz][c] * gy;
                        }
                    }
                    // stage y transposed (weights and -dt*grad_y folded into the tables)
#pragma unroll
                    for (int b = 0; b < M; ++b) {
                        const T wb = L.yt[BV][(ly * M + qy) * M + b];
                        const T wd = TW ? L.yt[BD][(ly * M + qy) * M + b] * cy : L.yt[BD][(ly * M + qy) * M + b];
#pragma unroll
                        for (int c = 0; c < M; ++c) {
                            K0[b][c] += wb * H0[c];
                            K0[b][c] += wd * Hy[c];
                            Kx[b][c] += wb * Hx[c];
                        }
                    }
                }
                // stage x transposed
#pragma unroll
                for (int a = 0; a < M; ++a) {
                    const T wb = L.xt[BV][(lx * M + qx) * M + a];
                    const T wd = TW ? L.xt[BD][(lx * M + qx) * M + a] * cx : L.xt[BD][(lx * M + qx) * M + a];
#pragma unroll
                    for (int b = 0; b < M; ++b)
#pragma unroll
                        for (int c = 0; c < M; ++c) {
                            if constexpr (FLUSH)
                                __hip_atomic_fetch_add(mine + c * PL + (lx + a) + BX * (ly + b),
                                                       static_cast<double>(wb * K0[b][c] + wd * Kx[b][c]),
                                                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
                            else {
                                R[FLUSH ? 0 : a][FLUSH ? 0 : b][FLUSH ? 0 : c] += wb * K0[b][c];
                                R[FLUSH ? 0 : a][FLUSH ? 0 : b][FLUSH ? 0 : c] += wd * Kx[b][c];
                            }
                        }
                }
            }
        }
    }
    if constexpr (!FLUSH && VAR != 4) {
#pragma unroll
        for (int c = 0; c < M; ++c)
#pragma unroll
            for (int b = 0; b < M; ++b)
#pragma unroll
                for (int a = 0; a < M; ++a)
                    __hip_atomic_fetch_add(mine + c * PL + (lx + a) + BX * (ly + b),
                                           static_cast<double>(R[FLUSH ? 0 : a][FLUSH ? 0 : b][FLUSH ? 0 : c]),
                                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
    }
}

// Stage the tile whose first element is o into B through registers: its coefficient block
// (zero outside the mesh) and its x and y tables, the backward ones weighted and with
// -dt*grad folded in.
template <int NTH = 0, typename T, int P, int TX, int TY, int TZ, bool KF>
__device__ __forceinline__ void rhs3_stage(rhs3_buf<T, P, TX, TY, TZ, KF>& B, tile3 o,
                                           const T* __restrict__ up, const dev_tables<T>& X,
                                           const dev_tables<T>& Y, int nz, const rhs_params<T>& prm,
                                           int tid) {
    using BUF = rhs3_buf<T, P, TX, TY, TZ, KF>;
    // NTH: threads of the workgroup (default one per element of the tile)
    constexpr int M = P + 1, NT = NTH ? NTH : TX * TY * TZ, BX = BUF::BX, BY = BUF::BY, NB = BUF::NB;
    static_assert(TX * M * M <= NT && TY * M * M <= NT, "one table entry per thread");
    const int nx = X.dofs, ny = Y.dofs;
    for (int i = tid; i < NB; i += NT) {
        const int bx = i % BX, r = i / BX, by = r % BY, bz = r / BY;
        const int gx = o.ex0 + bx, gy = o.ey0 + by, gz = o.ez0 + bz;
        const bool in = gx < nx && gy < ny && gz < nz;
        const long g = gx + static_cast<long>(nx) * (gy + static_cast<long>(ny) * gz);
        B.blk[i] = in ? up[g] : T(0);
        if constexpr (KF) B.kb[i] = in ? prm.kfield[g] : T(0);
    }
    const T cx = -prm.dt * prm.gx, cy = -prm.dt * prm.gy;
    if (tid < TX * M * M) {
        const int e = o.ex0 + tid / (M * M), q = (tid / M) % M;
        const bool in = e < X.elements;
        const T v = in ? X.val[static_cast<long>(o.ex0) * M * M + tid] : T(0);
        const T d = in ? X.der[static_cast<long>(o.ex0) * M * M + tid] : T(0);
        const T w = in ? X.wj[static_cast<long>(e) * M + q] : T(0);
        B.xt[FV][tid] = v;
        B.xt[FD][tid] = d;
        B.xt[BV][tid] = v * w;
        B.xt[BD][tid] = cx * (d * w);
    }
    if (tid < TY * M * M) {
        const int e = o.ey0 + tid / (M * M), q = (tid / M) % M;
        const bool in = e < Y.elements;
        const T v = in ? Y.val[static_cast<long>(o.ey0) * M * M + tid] : T(0);
        const T d = in ? Y.der[static_cast<long>(o.ey0) * M * M + tid] : T(0);
        const T w = in ? Y.wj[static_cast<long>(e) * M + q] : T(0);
        B.yt[FV][tid] = v;
        B.yt[FD][tid] = d;
        B.yt[BV][tid] = v * w;
        B.yt[BD][tid] = cy * (d * w);
    }
}

// s_waitcnt operand (gfx9 encoding: vmcnt bits 3:0 and 15:14, expcnt 6:4, lgkmcnt 11:8) that
// waits for every vector memory operation of the wave and for nothing else: vmcnt(0)
constexpr int kWaitVmem = 0x0F70;

// Copy n 32-bit words into LDS at dst (wave-uniform) from the global words src(k), k < n,
// with global-to-LDS loads, which use no registers and complete in the background: wave
// `wave` of NW takes the 64-word chunks wave, wave + NW, ...
template <int NW, typename F>
__device__ __forceinline__ void lds_fetch(uint32_t* dst, int n, int wave, int lane, F&& src) {
    for (int j = wave; j * 64 < n; j += NW) {
        const int k = j * 64 + lane;
        if (k < n) __builtin_amdgcn_global_load_lds(src(k), dst + j * 64, 4, 0, 0);
    }
}

// Start copying the tile whose first element is o into B: the coefficient block (indices
// outside the mesh clamped to the last DOF: those entries are read by no element of the
// mesh) and the tables as stored (zero-padded per tile; weighted, no -dt*grad).
template <typename T, int P, int TX, int TY, int TZ, bool KF>
__device__ __forceinline__ void rhs3_fetch(rhs3_buf<T, P, TX, TY, TZ, KF>& B, tile3 o,
                                           const T* __restrict__ up, const dev_tables<T>& X,
                                           const dev_tables<T>& Y, int nz, const rhs_params<T>& prm,
                                           int wave, int lane) {
    using BUF = rhs3_buf<T, P, TX, TY, TZ, KF>;
    constexpr int M = P + 1, NW = TZ, BX = BUF::BX, BY = BUF::BY, NB = BUF::NB;
    constexpr int DW = sizeof(T) / 4;  // words per value
    const int nx = X.dofs, ny = Y.dofs;
    auto block_word = [&](const T* base) {
        return [=](int k) {
            const int i = k / DW, r = i / BX;
            const int gx = min(o.ex0 + i % BX, nx - 1), gy = min(o.ey0 + r % BY, ny - 1);
            const int gz = min(o.ez0 + r / BY, nz - 1);
            const long g = gx + static_cast<long>(nx) * (gy + static_cast<long>(ny) * gz);
            return reinterpret_cast<const uint32_t*>(base + g) + k % DW;
        };
    };
    lds_fetch<NW>(reinterpret_cast<uint32_t*>(B.blk), NB * DW, wave, lane, block_word(up));
    if constexpr (KF)
        lds_fetch<NW>(reinterpret_cast<uint32_t*>(B.kb), NB * DW, wave, lane, block_word(prm.kfield));
    // the tables: one copy per table, each from a wave-uniform base
    const T* xs[4] = {X.val + static_cast<long>(o.ex0) * M * M, X.der + static_cast<long>(o.ex0) * M * M,
                      X.bval + static_cast<long>(o.ex0) * M * M, X.bder + static_cast<long>(o.ex0) * M * M};
    const T* ys[4] = {Y.val + static_cast<long>(o.ey0) * M * M, Y.der + static_cast<long>(o.ey0) * M * M,
                      Y.bval + static_cast<long>(o.ey0) * M * M, Y.bder + static_cast<long>(o.ey0) * M * M};
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const uint32_t* xw = reinterpret_cast<const uint32_t*>(xs[t]);
        const uint32_t* yw = reinterpret_cast<const uint32_t*>(ys[t]);
        lds_fetch<NW>(reinterpret_cast<uint32_t*>(B.xt[t]), TX * M * M * DW, wave, lane,
                      [=](int k) { return xw + k; });
        lds_fetch<NW>(reinterpret_cast<uint32_t*>(B.yt[t]), TY * M * M * DW, wave, lane,
                      [=](int k) { return yw + k; });
    }
}

// DOF plane k of the tile's block collects plane k - lz of the waves lz = k-P .. k; the sum
// goes to the rhs through the sink (rhs3_put).
template <bool ONE, typename T, int P, int TX, int TY, int TZ>
__device__ __forceinline__ void rhs3_add_block(const double* acc, tile3 o, const block_sink<T>& k,
                                               const rhs_params<T>& prm, int nx, int ny, int nz, int tid) {
    constexpr int M = P + 1, BX = TX + P, BY = TY + P, PL = BX * BY, NB = PL * (TZ + P);
    constexpr int NT = TX * TY * TZ;
    for (int i = tid; i < NB; i += NT) {
        const int bxy = i % PL, bz = i / PL;
        const int gx = o.ex0 + bxy % BX, gy = o.ey0 + bxy / BX, gz = o.ez0 + bz;
        double sum = 0;
#pragma unroll
        for (int d = 0; d < M; ++d) {
            const int w = bz - d;
            if (w >= 0 && w < TZ) sum += acc[(w * M + d) * PL + bxy];
        }
        if (gx < nx && gy < ny && gz < nz)
            rhs3_put<ONE, P, TX, TY, TZ>(k, prm, bxy % BX, bxy / BX, bz, gx, gy, gz,
                                         gx + static_cast<long>(nx) * (gy + static_cast<long>(ny) * gz), sum);
    }
}

// One workgroup per tile (block b -> tile by XCD-contiguous numbering): tiles of one colour,
// or (ONE) all ntx2 x nty2 x ntz tiles with the spill array prm.spill.
template <typename T, int P, int TX, int TY, int TZ, bool KF, int FM, int VAR, bool ONE>
__global__ __launch_bounds__(TX* TY* TZ, (rhs3_waves<T, P, VAR>())) void k_rhs3(
    const T* __restrict__ up, T* __restrict__ rhs, dev_tables<T> X, dev_tables<T> Y,
    dev_tables<T> Z, rhs_params<T> prm, int colour, int ntx2, int nty2) {
    constexpr int NT = TX * TY * TZ, NA = rhs3_acc_size<P, TX, TY, TZ>();
    static_assert(TX * TY == 64, "a wave must cover exactly one z-layer of the tile");
    __shared__ rhs3_lds<T, P, TX, TY, TZ, KF, 1> S;
    auto& L = S.b[0];
    double* acc = S.acc[0];

    const int tid = threadIdx.x;
    const int lx = tid % TX, ly = (tid / TX) % TY;
    const int lz = __builtin_amdgcn_readfirstlane(tid / (TX * TY));
    // Workgroups are dealt to the 8 XCDs round-robin; renumber them so that each XCD gets a
    // contiguous run of tiles (one slab of the domain), whose halos the next colour's launch
    // then finds in that XCD's L2.
    const int t = xcd_contiguous(blockIdx.x, gridDim.x);
    const tile3 o = rhs3_tile_of<ONE, TX, TY, TZ>(t, colour, ntx2, nty2);
    // the tile's DOF block (first(e) = e for these knot vectors: dof origin = element origin)
    rhs3_stage(L, o, up, X, Y, Z.dofs, prm, tid);
    for (int i = tid; i < NA; i += NT) acc[i] = 0.0;
    __syncthreads();
    T R[P + 1][P + 1][P + 1] = {};
    rhs3_element<T, P, TX, TY, TZ, KF, FM, VAR>(L, acc, X, Y, Z, prm, lx, ly, lz, o.ex0,
                                                      o.ey0, o.ez0, R);
    __syncthreads();
    const block_sink<T> sink = rhs3_sink<ONE, TX, TY, TZ>(rhs, o, X.elements, Y.elements, Z.elements);
    rhs3_add_block<ONE, T, P, TX, TY, TZ>(acc, o, sink, prm, X.dofs, Y.dofs, Z.dofs, tid);
}

// d/dk_b of w^T rhs(u; k) for one element of a 3D tile (lane lx, ly of wave lz; u in L.blk,
// w in L.kb), added to the wave's DOF planes as rhs3_element adds its contribution. The
// diffusion term of the element loop with a coefficient field (validation.hpp:110-115) is
// linear in k:  d/dk_b = -dt sum_e sum_q w_q J_e B_b(x_q) sum_d grad_d (d_d u)(d_d w).
// Sum-factorised: u, w and their x derivatives contracted along x for one x Gauss point at a
// time, then along y and z; the weighted product tested against the value tables, z, y, x.
// At p = 3 the element's block would not fit the registers: its part for each x point is
// added to the planes at once.
template <typename T, int P, int TX, int TY, int TZ>
__device__ __forceinline__ void kgrad3_element(const rhs3_buf<T, P, TX, TY, TZ, true>& L, double* acc,
                                               const dev_tables<T>& X, const dev_tables<T>& Y,
                                               const dev_tables<T>& Z, const rhs_params<T>& prm, int lx, int ly,
                                               int lz, int ex0, int ey0, int ez0) {
    using LDS = rhs3_buf<T, P, TX, TY, TZ, true>;
    constexpr int M = P + 1, BX = LDS::BX, BY = LDS::BY, PL = LDS::PL;
    constexpr bool FLUSH = P == 3;
    constexpr int RM = FLUSH ? 1 : M;
    const int ez = ez0 + lz;
    double* mine = acc + lz * M * PL;
    T R[RM][RM][RM];
#pragma unroll
    for (int a = 0; a < RM; ++a)
#pragma unroll
        for (int b = 0; b < RM; ++b)
#pragma unroll
            for (int c = 0; c < RM; ++c) R[a][b][c] = T(0);
    if (ez < Z.elements) {  // wave-uniform
        T Bz[M][M], Dz[M][M], wz[M];
        const T* zv = Z.val + static_cast<long>(ez) * M * M;
        const T* zd = Z.der + static_cast<long>(ez) * M * M;
#pragma unroll
        for (int q = 0; q < M; ++q) {
            wz[q] = uniform_load(Z.wj + static_cast<long>(ez) * M + q);
#pragma unroll
            for (int c = 0; c < M; ++c) {
                Bz[q][c] = uniform_load(zv + q * M + c);
                Dz[q][c] = uniform_load(zd + q * M + c);
            }
        }
        const T cx = -prm.dt * prm.gx, cy = -prm.dt * prm.gy, cz = -prm.dt * prm.gz;
        if (ex0 + lx < X.elements && ey0 + ly < Y.elements) {
#pragma unroll 1
            for (int qx = 0; qx < M; ++qx) {
                T bx[M], dx[M];
#pragma unroll
                for (int a = 0; a < M; ++a) {
                    bx[a] = L.xt[FV][(lx * M + qx) * M + a];
                    dx[a] = L.xt[FD][(lx * M + qx) * M + a];
                }
                T U0[M][M], U1[M][M], W0[M][M], W1[M][M];  // along x: value, x derivative
#pragma unroll
                for (int b = 0; b < M; ++b)
#pragma unroll
                    for (int c = 0; c < M; ++c) {
                        T u0 = 0, u1 = 0, w0 = 0, w1 = 0;
#pragma unroll
                        for (int a = 0; a < M; ++a) {
                            const int li = (lx + a) + BX * ((ly + b) + BY * (lz + c));
                            const T cu = L.blk[li], cw = L.kb[li];
                            u0 += bx[a] * cu;
                            u1 += dx[a] * cu;
                            w0 += bx[a] * cw;
                            w1 += dx[a] * cw;
                        }
                        U0[b][c] = u0;
                        U1[b][c] = u1;
                        W0[b][c] = w0;
                        W1[b][c] = w1;
                    }
                T K[M][M];
#pragma unroll
                for (int b = 0; b < M; ++b)
#pragma unroll
                    for (int c = 0; c < M; ++c) K[b][c] = T(0);
#pragma unroll 1
                for (int qy = 0; qy < M; ++qy) {
                    T by[M], dy[M];
#pragma unroll
                    for (int b = 0; b < M; ++b) {
                        by[b] = L.yt[FV][(ly * M + qy) * M + b];
                        dy[b] = L.yt[FD][(ly * M + qy) * M + b];
                    }
                    // along y: (value, value), (value, y derivative), (x derivative, value)
                    T u00[M], u01[M], u10[M], w00[M], w01[M], w10[M];
#pragma unroll
                    for (int c = 0; c < M; ++c) {
                        T s0 = 0, s1 = 0, s2 = 0, t0 = 0, t1 = 0, t2 = 0;
#pragma unroll
                        for (int b = 0; b < M; ++b) {
                            s0 += by[b] * U0[b][c];
                            s1 += dy[b] * U0[b][c];
                            s2 += by[b] * U1[b][c];
                            t0 += by[b] * W0[b][c];
                            t1 += dy[b] * W0[b][c];
                            t2 += by[b] * W1[b][c];
                        }
                        u00[c] = s0;
                        u01[c] = s1;
                        u10[c] = s2;
                        w00[c] = t0;
                        w01[c] = t1;
                        w10[c] = t2;
                    }
                    T H[M];
#pragma unroll
                    for (int c = 0; c < M; ++c) H[c] = T(0);
#pragma unroll
                    for (int qz = 0; qz < M; ++qz) {
                        T ux = 0, uy = 0, uz = 0, wx = 0, wy = 0, wv = 0;
#pragma unroll
                        for (int c = 0; c < M; ++c) {
                            ux += Bz[qz][c] * u10[c];
                            uy += Bz[qz][c] * u01[c];
                            uz += Dz[qz][c] * u00[c];
                            wx += Bz[qz][c] * w10[c];
                            wy += Bz[qz][c] * w01[c];
                            wv += Dz[qz][c] * w00[c];
                        }
                        const T g = wz[qz] * (cx * (ux * wx) + cy * (uy * wy) + cz * (uz * wv));
#pragma unroll
                        for (int c = 0; c < M; ++c) H[c] += Bz[qz][c] * g;
                    }
#pragma unroll
                    for (int b = 0; b < M; ++b) {
                        const T wb = L.yt[BV][(ly * M + qy) * M + b];
#pragma unroll
                        for (int c = 0; c < M; ++c) K[b][c] += wb * H[c];
                    }
                }
#pragma unroll
                for (int a = 0; a < M; ++a) {
                    const T wa = L.xt[BV][(lx * M + qx) * M + a];
#pragma unroll
                    for (int b = 0; b < M; ++b)
#pragma unroll
                        for (int c = 0; c < M; ++c) {
                            if constexpr (FLUSH)
                                __hip_atomic_fetch_add(mine + c * PL + (lx + a) + BX * (ly + b),
                                                       static_cast<double>(wa * K[b][c]), __ATOMIC_RELAXED,
                                                       __HIP_MEMORY_SCOPE_WAVEFRONT);
                            else
                                R[FLUSH ? 0 : a][FLUSH ? 0 : b][FLUSH ? 0 : c] += wa * K[b][c];
                        }
                }
            }
        }
    }
    if constexpr (!FLUSH) {
#pragma unroll
        for (int c = 0; c < M; ++c)
#pragma unroll
            for (int b = 0; b < M; ++b)
#pragma unroll
                for (int a = 0; a < M; ++a)
                    __hip_atomic_fetch_add(mine + c * PL + (lx + a) + BX * (ly + b),
                                           static_cast<double>(R[FLUSH ? 0 : a][FLUSH ? 0 : b][FLUSH ? 0 : c]),
                                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
    }
}

// The 3D k-field gradient over the tiles of the 3D element loop (k_rhs3's tile, staging and
// block write): u is staged as the coefficient block, w (prm.kfield) as the k block.
template <typename T, int P, int TX, int TY, int TZ, bool ONE>
__global__ __launch_bounds__(TX* TY* TZ) void k_kgrad3(const T* __restrict__ u, T* __restrict__ out,
                                                     dev_tables<T> X, dev_tables<T> Y, dev_tables<T> Z,
                                                     rhs_params<T> prm, int colour, int ntx2, int nty2) {
    constexpr int NT = TX * TY * TZ, NA = rhs3_acc_size<P, TX, TY, TZ>();
    static_assert(TX * TY == 64, "a wave must cover exactly one z-layer of the tile");
    __shared__ rhs3_lds<T, P, TX, TY, TZ, true, 1> S;
    auto& L = S.b[0];
    double* acc = S.acc[0];
    const int tid = threadIdx.x;
    const int lx = tid % TX, ly = (tid / TX) % TY;
    const int lz = __builtin_amdgcn_readfirstlane(tid / (TX * TY));
    const tile3 o = rhs3_tile_of<ONE, TX, TY, TZ>(xcd_contiguous(blockIdx.x, gridDim.x), colour, ntx2, nty2);
    rhs3_stage(L, o, u, X, Y, Z.dofs, prm, tid);
    for (int i = tid; i < NA; i += NT) acc[i] = 0.0;
    __syncthreads();
    kgrad3_element<T, P, TX, TY, TZ>(L, acc, X, Y, Z, prm, lx, ly, lz, o.ex0, o.ey0, o.ez0);
    __syncthreads();
    const block_sink<T> sink = rhs3_sink<ONE, TX, TY, TZ>(out, o, X.elements, Y.elements, Z.elements);
    rhs3_add_block<ONE, T, P, TX, TY, TZ>(acc, o, sink, prm, X.dofs, Y.dofs, Z.dofs, tid);
}

// Variant 3: two tiles per workgroup (tiles 2w, 2w+1 of the colour for workgroup w after
// XCD-contiguous renumbering). The second tile's data is copied into its own LDS buffer by
// global-to-LDS loads issued before the first tile's integration, so that its HBM/L2
// latency is hidden behind that work instead of stalling every workgroup at its start.
// Each tile has its own DOF planes and both are added to the rhs at the end: no global
// write precedes the integrations, so their z tables stay in scalar registers.
template <typename T, int P, int TX, int TY, int TZ, bool KF, int FM>
__global__ __launch_bounds__(TX* TY* TZ, 2) void k_rhs3_pipe(
    const T* __restrict__ up, T* __restrict__ rhs, dev_tables<T> X, dev_tables<T> Y,
    dev_tables<T> Z, rhs_params<T> prm, int colour, int ntx2, int nty2, int ntiles) {
    constexpr int NT = TX * TY * TZ, NA = rhs3_acc_size<P, TX, TY, TZ>();
    static_assert(TX * TY == 64, "a wave must cover exactly one z-layer of the tile");
    __shared__ rhs3_lds<T, P, TX, TY, TZ, KF, 2> S;
    auto& B0 = S.b[0];
    auto& B1 = S.b[1];
    double* acc0 = S.acc[0];
    double* acc1 = S.acc[1];

    const int tid = threadIdx.x, lane = tid % 64;
    const int lx = tid % TX, ly = (tid / TX) % TY;
    const int lz = __builtin_amdgcn_readfirstlane(tid / 64);
    const int w = xcd_contiguous(blockIdx.x, gridDim.x);
    const bool two = 2 * w + 1 < ntiles;  // uniform over the workgroup
    const tile3 o0 = rhs3_tile<TX, TY, TZ>(2 * w, colour, ntx2, nty2);
    const tile3 o1 = rhs3_tile<TX, TY, TZ>(two ? 2 * w + 1 : 2 * w, colour, ntx2, nty2);

    rhs3_fetch(B0, o0, up, X, Y, Z.dofs, prm, lz, lane);
    for (int i = tid; i < NA; i += NT) acc0[i] = acc1[i] = 0.0;
    __builtin_amdgcn_s_waitcnt(kWaitVmem);  // this wave's copies into B0 have landed
    __syncthreads();
    if (two) rhs3_fetch(B1, o1, up, X, Y, Z.dofs, prm, lz, lane);
    T R0[P + 1][P + 1][P + 1] = {};
    rhs3_element<T, P, TX, TY, TZ, KF, FM, 3>(B0, acc0, X, Y, Z, prm, lx, ly, lz, o0.ex0,
                                                    o0.ey0, o0.ez0, R0);
    if (two) {
        __builtin_amdgcn_s_waitcnt(kWaitVmem);  // the copies into B1
        __syncthreads();
        T R1[P + 1][P + 1][P + 1] = {};
        rhs3_element<T, P, TX, TY, TZ, KF, FM, 3>(B1, acc1, X, Y, Z, prm, lx, ly, lz, o1.ex0,
                                                        o1.ey0, o1.ez0, R1);
    }
    __syncthreads();
    const block_sink<T> sink = rhs3_sink<false, TX, TY, TZ>(rhs, o0, 0, 0, 0);
    rhs3_add_block<false, T, P, TX, TY, TZ>(acc0, o0, sink, prm, X.dofs, Y.dofs, Z.dofs, tid);
    if (two) rhs3_add_block<false, T, P, TX, TY, TZ>(acc1, o1, sink, prm, X.dofs, Y.dofs, Z.dofs, tid);
}

// Variant 4 (p <= 2): tiles of TX x TY x TZ elements with TZ/2 waves, wave w integrating the
// element layers 2w and 2w+1 one after the other. Their contributions share P of their P+1
// DOF planes, so the register block R is carried from the first layer to the second: after
// the first only its lowest plane is added to LDS, after the second all P+1 planes — P+1
// plane adds per two elements instead of 2(P+1) (a third fewer LDS adds at p = 2), and the
// taller tile re-reads fewer halo planes. Wave w owns the LDS planes of DOF planes 2w ..
// 2w+P+1; the block add, the colouring and the one-launch tiling are those of the other
// variants.
template <typename T, int P, int TX, int TY, int TZ, bool KF, int FM>
__global__ __launch_bounds__(TX* TY*(TZ / 2), 2) void k_rhs3_zpair(
    const T* __restrict__ up, T* __restrict__ rhs, dev_tables<T> X, dev_tables<T> Y,
    dev_tables<T> Z, rhs_params<T> prm, int colour, int ntx2, int nty2) {
    constexpr int M = P + 1, NW = TZ / 2, NT = TX * TY * NW, BX = TX + P, BY = TY + P;
    constexpr int PL = BX * BY, NB = PL * (TZ + P), WP = P + 2;  // WP: planes per wave
    static_assert(TX * TY == 64 && TZ % 2 == 0 && TZ >= P, "one wave per pair of layers");
    struct lds_t {
        rhs3_buf<T, P, TX, TY, TZ, KF> b;
        double acc[NW * WP * PL];
    };
    __shared__ lds_t S;

    const int tid = threadIdx.x;
    const int lx = tid % TX, ly = (tid / TX) % TY;
    const int w = __builtin_amdgcn_readfirstlane(tid / 64);
    const int t = xcd_contiguous(blockIdx.x, gridDim.x);
    const tile3 o = rhs3_tile<TX, TY, TZ>(t, colour, ntx2, nty2);
    rhs3_stage<NT>(S.b, o, up, X, Y, Z.dofs, prm, tid);
    for (int i = tid; i < NW * WP * PL; i += NT) S.acc[i] = 0.0;
    __syncthreads();

    double* mine = S.acc + w * WP * PL;
    T R[M][M][M] = {};
    rhs3_element<T, P, TX, TY, TZ, KF, FM, 4>(S.b, mine, X, Y, Z, prm, lx, ly, 2 * w, o.ex0,
                                                    o.ey0, o.ez0, R);
#pragma unroll
    for (int b = 0; b < M; ++b)
#pragma unroll
        for (int a = 0; a < M; ++a) {  // the first layer's lowest plane is complete
            __hip_atomic_fetch_add(mine + (lx + a) + BX * (ly + b), static_cast<double>(R[a][b][0]),
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
#pragma unroll
            for (int c = 0; c < P; ++c) R[a][b][c] = R[a][b][c + 1];
            R[a][b][P] = T(0);
        }
    rhs3_element<T, P, TX, TY, TZ, KF, FM, 4>(S.b, mine, X, Y, Z, prm, lx, ly, 2 * w + 1,
                                                    o.ex0, o.ey0, o.ez0, R);
#pragma unroll
    for (int c = 0; c < M; ++c)
#pragma unroll
        for (int b = 0; b < M; ++b)
#pragma unroll
            for (int a = 0; a < M; ++a)
                __hip_atomic_fetch_add(mine + (1 + c) * PL + (lx + a) + BX * (ly + b),
                                       static_cast<double>(R[a][b][c]), __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_WAVEFRONT);
    __syncthreads();
    // DOF plane k of the block collects plane k - 2w of the waves w with 0 <= k - 2w <= P+1
    const block_sink<T> sink = rhs3_sink<false, TX, TY, TZ>(rhs, o, 0, 0, 0);
    for (int i = tid; i < NB; i += NT) {
        const int bxy = i % PL, bz = i / PL;
        const int gx = o.ex0 + bxy % BX, gy = o.ey0 + bxy / BX, gz = o.ez0 + bz;
        double sum = 0;
#pragma unroll
        for (int ww = 0; ww < NW; ++ww) {
            const int pl = bz - 2 * ww;
            if (pl >= 0 && pl < WP) sum += S.acc[(ww * WP + pl) * PL + bxy];
        }
        if (gx < X.dofs && gy < Y.dofs && gz < Z.dofs)
            rhs3_put<false, P, TX, TY, TZ>(sink, prm, bxy % BX, bxy / BX, bz, gx, gy, gz,
                                         gx + static_cast<long>(X.dofs) * (gy + static_cast<long>(Y.dofs) * gz), sum);
    }
}

// ------------------------------------------------------------------------------------
// element-loop RHS, 2D
// ------------------------------------------------------------------------------------
// The end of a 2D tile (TX x TY elements, tile (tx, ty)): the element blocks R of its lanes
// (lane = element (tid % TX, tid / TX)) are added per wave into the wave's DOF rows of acc
// (zeroed by the caller before its first barrier; wave w holds element rows w*WY.. and DOF
// rows w*WY .. w*WY+WR-1), and after one barrier the tile's DOF block is added into rhs, or
// (ONE) its owned entries go to rhs and the others to the spill arrays of prm.
template <typename T, int P, int TX, int TY, bool ONE>
__device__ __forceinline__ void rhs2_flush(const T (&R)[P + 1][P + 1], double* __restrict__ acc, T* __restrict__ rhs,
                                           const dev_tables<T>& X, const dev_tables<T>& Y, const rhs_params<T>& prm,
                                           int tx, int ty) {
    constexpr int M = P + 1, NT = TX * TY;
    constexpr int BX = TX + P, BY = TY + P, NB = BX * BY;
    constexpr int WY = 64 / TX, NW = NT / 64, WR = WY + P;
    const int tid = threadIdx.x;
    const int lx = tid % TX, ly = tid / TX;
    const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const int wy = ly - wave * WY;  // element row inside the wave
    const int ex0 = tx * TX, ey0 = ty * TY;
    const int nx = X.dofs, ny = Y.dofs;
    double* mine = acc + wave * WR * BX;
#pragma unroll
    for (int b = 0; b < M; ++b)
#pragma unroll
        for (int a = 0; a < M; ++a)
            __hip_atomic_fetch_add(mine + (wy + b) * BX + lx + a, static_cast<double>(R[a][b]),
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
    __syncthreads();

    const bool lastx = ex0 + TX >= X.elements, lasty = ey0 + TY >= Y.elements;
    for (int i = tid; i < NB; i += NT) {
        const int bx = i % BX, by = i / BX;
        const int gx = ex0 + bx, gy = ey0 + by;
        if (gx >= nx || gy >= ny) continue;
        double sum = 0;
        for (int w = 0; w < NW; ++w) {
            const int r = by - w * WY;
            if (r >= 0 && r < WR) sum += acc[(w * WR + r) * BX + bx];
        }
        const long g = gx + static_cast<long>(nx) * gy;
        if constexpr (ONE) {
            const int dx = bx >= TX && !lastx, dy = by >= TY && !lasty;
            if (!(dx | dy)) {
                rhs[g] = prm.store ? static_cast<T>(sum) : rhs[g] + static_cast<T>(sum);
            } else {
                const int cx = dx ? (tx + 1) * P + bx - TX : gx;
                const int cy = dy ? (ty + 1) * P + by - TY : gy;
                prm.spill[spill_index(prm, dx, dy, 0, cx, cy, 0)] = static_cast<T>(sum);
            }
        } else if (prm.store) {
            // colour launches on an rhs without a start value: the first colour to reach a DOF
            // stores. Another tile holds the entry in x when bx < P (tile tx - 1) or bx >= TX
            // (tile tx + 1), in y likewise; those tiles' colours flip the parity bits, and the
            // colours run in the order 0, 1, 2, 3.
            const int c = (tx & 1) | ((ty & 1) << 1);
            const bool hx = (bx < P && tx > 0) || (bx >= TX && !lastx);
            const bool hy = (by < P && ty > 0) || (by >= TY && !lasty);
            const bool first = (!hx || !(c & 1)) && (!hy || !(c & 2));
            rhs[g] = first ? static_cast<T>(sum) : rhs[g] + static_cast<T>(sum);
        } else {
            rhs[g] += static_cast<T>(sum);
        }
    }
}

// One tile of TX x TY elements, tile t of the given parity colour (ntx2 tiles of that colour
// per tile row), added into rhs; or (ONE) tile t of all tiles (ntx2 of them per tile row),
// whose owned DOF-block entries go to the rhs and the others to the spill arrays of prm
// (rhs3_put's ownership and layout, in two directions): the batches' 8 x 8 tiles and the
// adjoint pair; the element loop of one problem runs in strips (adsg_rhs2_march.hip). The LDS arrays are separate
// __shared__ objects: gathered into one struct, the compiler read the tables with
// ds_read2_b64 pairs instead of ds_read_b128 and the p = 3 batch kernel ran 1.5x slower.
template <typename T, int P, int TX, int TY, bool KF, bool ONE>
__device__ __forceinline__ void rhs2_tile(const T* __restrict__ up, T* __restrict__ rhs, const dev_tables<T>& X,
                                          const dev_tables<T>& Y, const rhs_params<T>& prm, int colour, int t,
                                          int ntx2) {
    constexpr int M = P + 1, NT = TX * TY;
    constexpr int BX = TX + P, BY = TY + P, NB = BX * BY;
    constexpr int WY = 64 / TX;  // element rows per wave
    constexpr int NW = NT / 64;  // waves
    constexpr int WR = WY + P;   // DOF rows touched by one wave
    static_assert(TX <= 64 && 64 % TX == 0 && TY % WY == 0, "waves must cover whole element rows");
    __shared__ T blk[NB];
    __shared__ T kb[KF ? NB : 1];
    __shared__ T fvx[TX * M * M], fdx[TX * M * M], bvx[TX * M * M], bdx[TX * M * M];
    __shared__ T fvy[TY * M * M], fdy[TY * M * M], bvy[TY * M * M], bdy[TY * M * M];
    __shared__ double acc[NW * WR * BX];  // wave w owns DOF rows w*WY .. w*WY+WR-1

    const int tid = threadIdx.x;
    const int tx = ONE ? t % ntx2 : 2 * (t % ntx2) + (colour & 1);
    const int ty = ONE ? t / ntx2 : 2 * (t / ntx2) + ((colour >> 1) & 1);
    const int ex0 = tx * TX, ey0 = ty * TY;
    const int nx = X.dofs, ny = Y.dofs;

    for (int i = tid; i < NB; i += NT) {
        const int bx = i % BX, by = i / BX;
        const int gx = ex0 + bx, gy = ey0 + by;
        const bool in = gx < nx && gy < ny;
        const long g = gx + static_cast<long>(nx) * gy;
        blk[i] = in ? up[g] : T(0);
        if constexpr (KF) kb[i] = in ? prm.kfield[g] : T(0);
    }
    const T cx = -prm.dt * prm.gx, cy = -prm.dt * prm.gy;
    for (int i = tid; i < TX * M * M; i += NT) {
        const int e = ex0 + i / (M * M), q = (i / M) % M;
        const bool in = e < X.elements;
        const T v = in ? X.val[static_cast<long>(ex0) * M * M + i] : T(0);
        const T d = in ? X.der[static_cast<long>(ex0) * M * M + i] : T(0);
        const T w = in ? X.wj[static_cast<long>(e) * M + q] : T(0);
        fvx[i] = v;
        fdx[i] = d;
        bvx[i] = v * w;
        bdx[i] = cx * (d * w);
    }
    for (int i = tid; i < TY * M * M; i += NT) {
        const int e = ey0 + i / (M * M), q = (i / M) % M;
        const bool in = e < Y.elements;
        const T v = in ? Y.val[static_cast<long>(ey0) * M * M + i] : T(0);
        const T d = in ? Y.der[static_cast<long>(ey0) * M * M + i] : T(0);
        const T w = in ? Y.wj[static_cast<long>(e) * M + q] : T(0);
        fvy[i] = v;
        fdy[i] = d;
        bvy[i] = v * w;
        bdy[i] = d * w;
    }
    for (int i = tid; i < NW * WR * BX; i += NT) acc[i] = 0.0;
    __syncthreads();

    const int lx = tid % TX, ly = tid / TX;
    T R[M][M];
#pragma unroll
    for (int a = 0; a < M; ++a)
#pragma unroll
        for (int b = 0; b < M; ++b) R[a][b] = T(0);
    if (ex0 + lx < X.elements && ey0 + ly < Y.elements) {
        T By[M][M], Dy[M][M];
#pragma unroll
        for (int q = 0; q < M; ++q)
#pragma unroll
            for (int b = 0; b < M; ++b) {
                By[q][b] = fvy[(ly * M + q) * M + b];
                Dy[q][b] = fdy[(ly * M + q) * M + b];
            }
        const T mass = prm.mass;
#pragma unroll
        for (int qx = 0; qx < M; ++qx) {
            T bx[M], dx[M];
#pragma unroll
            for (int a = 0; a < M; ++a) {
                bx[a] = fvx[(lx * M + qx) * M + a];
                dx[a] = fdx[(lx * M + qx) * M + a];
            }
            T A0[M], A1[M], KA[KF ? M : 1];
#pragma unroll
            for (int b = 0; b < M; ++b) {
                T s0 = 0, s1 = 0, sk = 0;
#pragma unroll
                for (int a = 0; a < M; ++a) {
                    const int li = (lx + a) + BX * (ly + b);
                    const T cv = blk[li];
                    s0 += bx[a] * cv;
                    s1 += dx[a] * cv;
                    if constexpr (KF) sk += bx[a] * kb[li];
                }
                A0[b] = s0;
                A1[b] = s1;
                if constexpr (KF) KA[b] = sk;
            }
            T K0[M], Kx[M];
#pragma unroll
            for (int b = 0; b < M; ++b) K0[b] = Kx[b] = T(0);
#pragma unroll
            for (int qy = 0; qy < M; ++qy) {
                T u = 0, uy = 0, ux = 0, kv = 0;
#pragma unroll
                for (int b = 0; b < M; ++b) {
                    u += By[qy][b] * A0[b];
                    uy += Dy[qy][b] * A0[b];
                    ux += By[qy][b] * A1[b];
                    if constexpr (KF) kv += By[qy][b] * KA[b];
                }
                T g0 = mass * u;
                if (prm.reaction != T(0)) g0 += prm.dt * prm.reaction * u * (T(1) - u);
                T gx = ux, gy = cy * uy;
                if constexpr (KF) {
                    gx *= kv;
                    gy *= kv;
                }
                // stage y transposed (weights folded into the backward y tables)
#pragma unroll
                for (int b = 0; b < M; ++b) {
                    const T wb = bvy[(ly * M + qy) * M + b], wd = bdy[(ly * M + qy) * M + b];
                    K0[b] += wb * g0;
                    K0[b] += wd * gy;
                    Kx[b] += wb * gx;
                }
            }
#pragma unroll
            for (int a = 0; a < M; ++a) {
                const T wb = bvx[(lx * M + qx) * M + a], wd = bdx[(lx * M + qx) * M + a];
#pragma unroll
                for (int b = 0; b < M; ++b) {
                    R[a][b] += wb * K0[b];
                    R[a][b] += wd * Kx[b];
                }
            }
        }
    }
    rhs2_flush<T, P, TX, TY, ONE>(R, acc, rhs, X, Y, prm, tx, ty);
}

// d/dk_b of w^T rhs(u; k) over one 2D tile (the tile of rhs2_tile for colour, t, ntx2),
// added into out like rhs2_tile adds its blocks. The diffusion term of the element loop
// (validation.hpp:110-115 with a coefficient field) is linear in k, so
//   d/dk_b = -dt sum_e sum_q w_q J_e B_b(x_q) (gx u_x w_x + gy u_y w_y)(x_q).
// Per element: u and w and their x derivatives contracted along x for one x Gauss point at a
// time, then along y for each y point; the weighted product g tested against the value
// tables, y then x (the weights folded into the backward tables).
template <typename T, int P, int TX, int TY, bool ONE>
__device__ __forceinline__ void kgrad2_tile(const T* __restrict__ u, const T* __restrict__ w, T* __restrict__ out,
                                            const dev_tables<T>& X, const dev_tables<T>& Y, const rhs_params<T>& prm,
                                            int colour, int t, int ntx2) {
    constexpr int M = P + 1, NT = TX * TY;
    constexpr int BX = TX + P, BY = TY + P, NB = BX * BY;
    constexpr int WY = 64 / TX, NW = NT / 64, WR = WY + P;
    static_assert(TX <= 64 && 64 % TX == 0 && TY % WY == 0, "waves must cover whole element rows");
    __shared__ T ub[NB], wb[NB];
    __shared__ T fvx[TX * M * M], fdx[TX * M * M], bvx[TX * M * M];
    __shared__ T fvy[TY * M * M], fdy[TY * M * M], bvy[TY * M * M];
    __shared__ double acc[NW * WR * BX];

    const int tid = threadIdx.x;
    const int tx = ONE ? t % ntx2 : 2 * (t % ntx2) + (colour & 1);
    const int ty = ONE ? t / ntx2 : 2 * (t / ntx2) + ((colour >> 1) & 1);
    const int ex0 = tx * TX, ey0 = ty * TY;
    const int nx = X.dofs, ny = Y.dofs;
    for (int i = tid; i < NB; i += NT) {
        const int gx = ex0 + i % BX, gy = ey0 + i / BX;
        const bool in = gx < nx && gy < ny;
        const long g = gx + static_cast<long>(nx) * gy;
        ub[i] = in ? u[g] : T(0);
        wb[i] = in ? w[g] : T(0);
    }
    for (int i = tid; i < TX * M * M; i += NT) {
        const int e = ex0 + i / (M * M), q = (i / M) % M;
        const bool in = e < X.elements;
        const T v = in ? X.val[static_cast<long>(ex0) * M * M + i] : T(0);
        fvx[i] = v;
        fdx[i] = in ? X.der[static_cast<long>(ex0) * M * M + i] : T(0);
        bvx[i] = v * (in ? X.wj[static_cast<long>(e) * M + q] : T(0));
    }
    for (int i = tid; i < TY * M * M; i += NT) {
        const int e = ey0 + i / (M * M), q = (i / M) % M;
        const bool in = e < Y.elements;
        const T v = in ? Y.val[static_cast<long>(ey0) * M * M + i] : T(0);
        fvy[i] = v;
        fdy[i] = in ? Y.der[static_cast<long>(ey0) * M * M + i] : T(0);
        bvy[i] = v * (in ? Y.wj[static_cast<long>(e) * M + q] : T(0));
    }
    for (int i = tid; i < NW * WR * BX; i += NT) acc[i] = 0.0;
    __syncthreads();

    const int lx = tid % TX, ly = tid / TX;
    const T cx = -prm.dt * prm.gx, cy = -prm.dt * prm.gy;
    T R[M][M];
#pragma unroll
    for (int a = 0; a < M; ++a)
#pragma unroll
        for (int b = 0; b < M; ++b) R[a][b] = T(0);
    if (ex0 + lx < X.elements && ey0 + ly < Y.elements) {
        T By[M][M], Dy[M][M];
#pragma unroll
        for (int q = 0; q < M; ++q)
#pragma unroll
            for (int b = 0; b < M; ++b) {
                By[q][b] = fvy[(ly * M + q) * M + b];
                Dy[q][b] = fdy[(ly * M + q) * M + b];
            }
#pragma unroll
        for (int qx = 0; qx < M; ++qx) {
            T bx[M], dx[M];
#pragma unroll
            for (int a = 0; a < M; ++a) {
                bx[a] = fvx[(lx * M + qx) * M + a];
                dx[a] = fdx[(lx * M + qx) * M + a];
            }
            T U0[M], U1[M], W0[M], W1[M];  // along x: value and x derivative, per DOF row b
#pragma unroll
            for (int b = 0; b < M; ++b) {
                T u0 = 0, u1 = 0, w0 = 0, w1 = 0;
#pragma unroll
                for (int a = 0; a < M; ++a) {
                    const int li = (lx + a) + BX * (ly + b);
                    const T cu = ub[li], cw = wb[li];
                    u0 += bx[a] * cu;
                    u1 += dx[a] * cu;
                    w0 += bx[a] * cw;
                    w1 += dx[a] * cw;
                }
                U0[b] = u0;
                U1[b] = u1;
                W0[b] = w0;
                W1[b] = w1;
            }
            T K[M];
#pragma unroll
            for (int b = 0; b < M; ++b) K[b] = T(0);
#pragma unroll
            for (int qy = 0; qy < M; ++qy) {
                T ux = 0, uy = 0, wx = 0, wy = 0;
#pragma unroll
                for (int b = 0; b < M; ++b) {
                    ux += By[qy][b] * U1[b];
                    uy += Dy[qy][b] * U0[b];
                    wx += By[qy][b] * W1[b];
                    wy += Dy[qy][b] * W0[b];
                }
                const T g = cx * (ux * wx) + cy * (uy * wy);
#pragma unroll
                for (int b = 0; b < M; ++b) K[b] += bvy[(ly * M + qy) * M + b] * g;
            }
#pragma unroll
            for (int a = 0; a < M; ++a) {
                const T wa = bvx[(lx * M + qx) * M + a];
#pragma unroll
                for (int b = 0; b < M; ++b) R[a][b] += wa * K[b];
            }
        }
    }
    rhs2_flush<T, P, TX, TY, ONE>(R, acc, out, X, Y, prm, tx, ty);
}

template <typename T, int P, int TX, int TY, bool ONE>
__global__ __launch_bounds__(TX* TY) void k_kgrad2(const T* __restrict__ u, const T* __restrict__ w,
                                                   T* __restrict__ out, dev_tables<T> X, dev_tables<T> Y,
                                                   rhs_params<T> prm, int colour, int ntx2) {
    kgrad2_tile<T, P, TX, TY, ONE>(u, w, out, X, Y, prm, colour, xcd_contiguous(blockIdx.x, gridDim.x), ntx2);
}

// The 2D adjoint step's two element passes in one launch over all tiles (one-launch tiling):
// blocks [0, tiles) the element loop of the form for w (rhs2_tile, into out_r, prm_r), blocks
// [tiles, 2 tiles) the k-field gradient of u and w (kgrad2_tile, into out_k, prm_k), each
// with its own spill arrays; the two halves share nothing, and twice the blocks fill more of
// the device than either pass alone on small meshes.
template <typename T, int P, int TX, int TY>
__global__ __launch_bounds__(TX* TY) void k_adjoint2(const T* __restrict__ w, const T* __restrict__ u,
                                                     T* __restrict__ out_r, T* __restrict__ out_k, dev_tables<T> X,
                                                     dev_tables<T> Y, rhs_params<T> prm_r, rhs_params<T> prm_k,
                                                     int ntx, int tiles) {
    const int b = static_cast<int>(blockIdx.x);
    if (b < tiles)
        rhs2_tile<T, P, TX, TY, true, true>(w, out_r, X, Y, prm_r, 0, b, ntx);
    else
        kgrad2_tile<T, P, TX, TY, true>(u, w, out_k, X, Y, prm_k, 0, b - tiles, ntx);
}

// Many 2D problems of degree P in one launch per parity colour: block b belongs to the last
// item whose first[colour] <= b (items in problem order), and is tile b - first[colour] of
// it. (The other choice of batched element kernel: the strips of adsg_rhs2_march.hip.)
template <typename T, int P, int TX>
__global__ __launch_bounds__(TX* TX) void k_rhs2_batch(const rhs2_item<T>* __restrict__ items, int nitems,
                                                       int colour) {
    const int b = xcd_contiguous(blockIdx.x, gridDim.x);
    int lo = 0, hi = nitems - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) / 2;
        if (items[mid].first[colour] <= b)
            lo = mid;
        else
            hi = mid - 1;
    }
    const rhs2_item<T>& it = items[lo];
    rhs2_tile<T, P, TX, TX, false, false>(it.up, it.rhs, it.X, it.Y, it.prm, colour, b - it.first[colour],
                                                 it.ntx2[colour]);
}

// tile shapes (elements) per dimension and degree: one lane per element
template <int D, int P>
struct tile;
template <int P>
struct tile<2, P> {
    static constexpr int X = 16, Y = 16, Z = 1;
};
template <>
struct tile<3, 1> {
    static constexpr int X = 8, Y = 8, Z = 4;
};
template <>
struct tile<3, 2> {
    static constexpr int X = 8, Y = 8, Z = 4;
};
template <>
struct tile<3, 3> {
    static constexpr int X = 8, Y = 8, Z = 3;
};

template <typename T, int P, bool KF, int FM, int VAR>
hipError_t rhs3_colours(const T* up, T* rhs, const dev_tables<T>* d, const rhs_params<T>& prm,
                        hipStream_t s) {
    using TL = tile<3, P>;
    const int ntx = (d[0].elements + TL::X - 1) / TL::X;
    const int nty = (d[1].elements + TL::Y - 1) / TL::Y;
    const int ntz = (d[2].elements + TL::Z - 1) / TL::Z;
    constexpr int NT = TL::X * TL::Y * TL::Z;
    for (int c = 0; c < 8; ++c) {
        const int cx = c & 1, cy = (c >> 1) & 1, cz = (c >> 2) & 1;
        const int nx2 = (ntx - cx + 1) / 2, ny2 = (nty - cy + 1) / 2, nz2 = (ntz - cz + 1) / 2;
        const long tiles = static_cast<long>(nx2) * ny2 * nz2;
        if (tiles == 0) continue;
        if constexpr (VAR == 4 && P <= 2) {
            // tiles twice as tall (2 TL::Z element layers), TL::Z waves
            constexpr int TZ2 = 2 * TL::Z;
            const int ntz2 = (d[2].elements + TZ2 - 1) / TZ2, nz22 = (ntz2 - cz + 1) / 2;
            const long tiles2 = static_cast<long>(nx2) * ny2 * nz22;
            if (tiles2 > 0)
                hipLaunchKernelGGL((k_rhs3_zpair<T, P, TL::X, TL::Y, TZ2, KF, FM>), dim3(tiles2),
                                   dim3(NT), 0, s, up, rhs, d[0], d[1], d[2], prm, c, nx2, ny2);
        } else if constexpr (VAR == 3) {
            hipLaunchKernelGGL((k_rhs3_pipe<T, P, TL::X, TL::Y, TL::Z, KF, FM>),
                               dim3((tiles + 1) / 2), dim3(NT), 0, s, up, rhs, d[0], d[1], d[2], prm,
                               c, nx2, ny2, static_cast<int>(tiles));
        } else {
            // variant 4 at p = 3 (its register block would spill) runs as variant 2
            constexpr int V = VAR == 4 ? 2 : VAR;
            hipLaunchKernelGGL((k_rhs3<T, P, TL::X, TL::Y, TL::Z, KF, FM, V, false>), dim3(tiles),
                               dim3(NT), 0, s, up, rhs, d[0], d[1], d[2], prm, c, nx2, ny2);
        }
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// describes the fix-up of a one-launch element loop (layout of q) for a later kernel
template <typename T>
void defer_fixup(rhs_fixup<T>& fx, const rhs_params<T>& q, int p, const int tile[3], const int nt[3],
                 const int n[3]) {
    fx.spill = q.spill;
    for (int k = 0; k < 8; ++k) fx.off[k] = q.spill_off[k];
    for (int d = 0; d < 3; ++d) {
        fx.ext[d][0] = q.spill_ext[d][0];
        fx.ext[d][1] = q.spill_ext[d][1];
        fx.tile[d] = tile[d];
        fx.nt[d] = nt[d];
        fx.n[d] = n[d];
    }
    fx.p = p;
}

// A deferred fix-up over the DOFs (nx x ny x nz; nz = 1 in 2D): the spill sum of every DOF
// that has one, then the boundary zeroing (k_zero_boundary's, when asked for), in one pass.
// Tile t_d - 1 of a direction holds an entry for DOF g in its top P layers when l_d < P and
// t_d > 0 (t_d = min(g_d / tile_d, nt_d - 1), l_d = g_d - tile_d t_d): up to 7 entries, of the
// earlier tiles in some of the directions, added in the order delta = 1..7 as double.
// A wave takes a row of DOFs along x, so that everything that depends on y and z is scalar (a
// lane per DOF spent the pass on 64-bit index arithmetic and divisions, FP32 as long as FP64:
// 130^3 p = 2 12.8 us, 195^3 p = 3 39.5 us FP64 and 37 FP32, here 11.7, 30.4 and 25), and all
// loads of 64 DOFs are issued before the first is used: lanes without an entry read entry 0.
// (The passes of a row in flight together gained nothing.)
template <typename T, bool Y, bool Z>
__device__ __forceinline__ void rhs_fixup_row(T* __restrict__ out, const rhs_fixup<T>& fx, const T* const (&e)[8]) {
    const int lane = threadIdx.x & 63, nx = fx.n[0], P = fx.p;
    for (int x0 = 0; x0 < nx; x0 += 64) {
        const int gx = min(x0 + lane, nx - 1);
        const int tx = min(static_cast<int>(static_cast<unsigned>(gx) / static_cast<unsigned>(fx.tile[0])), fx.nt[0] - 1);
        const int lx = gx - fx.tile[0] * tx;
        const bool sx = lx < P && tx > 0;
        const int hx = sx ? tx * P + lx : 0;
        T v[8];
#pragma unroll
        for (int d = 1; d < 8; ++d) {
            if (((d & 2) && !Y) || ((d & 4) && !Z)) continue;
            v[d] = e[d][(d & 1) ? hx : gx];
        }
        const T r = out[gx];
        double sum = 0;
#pragma unroll
        for (int d = 1; d < 8; ++d) {
            if (((d & 2) && !Y) || ((d & 4) && !Z)) continue;
            sum += (d & 1) && !sx ? 0.0 : static_cast<double>(v[d]);
        }
        const bool zero = fx.zero_boundary && (gx == 0 || gx == nx - 1);
        if (x0 + lane < nx && (Y || Z || sx || zero)) out[gx] = zero ? T(0) : r + static_cast<T>(sum);
    }
}

// rows of DOFs per workgroup of a fix-up, one per wave
constexpr int kFixupRows = 4;
// Many short rows take a lane per DOF instead: a row costs 0.4 to 0.5 ns whatever its length (400
// x 400 rows 62 to 70 us, a lane per DOF 5 to 20 of them up to 16 DOFs; 130 x 130 rows of 3 / 24 /
// 48 / 64 DOFs, p = 1: 9.2 / 8.7 / 9.0 / 9.4 against 3.4 / 5.6 / 7.7 / 9.1 us, p = 3 9.1 / 9.4 /
// 9.8 / 9.9 against 4.5 / 6.4 / 9.7 / 10.8; of 48 x 48 rows 3.4 to 4.7 against 3.4 to 4.9).
constexpr int kFixupRowLength = 56;
constexpr long kFixupManyRows = 8192;
constexpr unsigned kFixupBlocks = 1u << 23;  // workgroups per launch: a grid has fewer than 2^32 lanes

template <typename T>
__device__ __forceinline__ void rhs_fixup_block(T* __restrict__ rhs, const rhs_fixup<T>& fx, unsigned block) {
    const unsigned ny = fx.n[1], row = block * kFixupRows + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (row >= ny * static_cast<unsigned>(fx.n[2])) return;
    const int gz = static_cast<int>(row / ny), gy = static_cast<int>(row - gz * ny), nx = fx.n[0], P = fx.p;
    T* out = rhs + static_cast<long>(row) * nx;
    const bool edge = gy == 0 || gy == fx.n[1] - 1 || (fx.n[2] > 1 && (gz == 0 || gz == fx.n[2] - 1));
    if (fx.zero_boundary && (edge || !fx.spill)) {
        for (int x = threadIdx.x & 63; x < nx; x += 64)
            if (edge || x == 0 || x == nx - 1) out[x] = T(0);
        return;
    }
    if (!fx.spill) return;
    const int ty = min(gy / fx.tile[1], fx.nt[1] - 1), tz = min(gz / fx.tile[2], fx.nt[2] - 1);
    const int ly = gy - fx.tile[1] * ty, lz = gz - fx.tile[2] * tz;
    const T* e[8];  // the row's entries in each spill array
    e[0] = nullptr;
#pragma unroll
    for (int d = 1; d < 8; ++d) {
        const int dx = d & 1, dy = (d >> 1) & 1, dz = d >> 2;
        e[d] = fx.spill + fx.off[d] +
               static_cast<long>(fx.ext[0][dx]) *
                   ((dy ? ty * P + ly : gy) + static_cast<long>(fx.ext[1][dy]) * (dz ? tz * P + lz : gz));
    }
    const bool sy = ly < P && ty > 0, sz = lz < P && tz > 0;
    if (sy && sz)
        rhs_fixup_row<T, true, true>(out, fx, e);
    else if (sy)
        rhs_fixup_row<T, true, false>(out, fx, e);
    else if (sz)
        rhs_fixup_row<T, false, true>(out, fx, e);
    else
        rhs_fixup_row<T, false, false>(out, fx, e);
}

template <typename T>
__global__ __launch_bounds__(64 * kFixupRows) void k_rhs_fixup(T* __restrict__ rhs, rhs_fixup<T> fx,
                                                               unsigned first) {
    rhs_fixup_block<T>(rhs, fx, first + blockIdx.x);
}

// A lane per DOF, for short rows (launch_rhs_fixup): the same sums in the same order.
template <typename T>
__global__ __launch_bounds__(256) void k_rhs_fixup_dofs(T* __restrict__ rhs, rhs_fixup<T> fx, unsigned N) {
    const unsigned g = blockIdx.x * 256 + threadIdx.x, nx = fx.n[0], ny = fx.n[1];
    if (g >= N) return;
    const unsigned row = g / nx, plane = row / ny;
    const int gx = static_cast<int>(g - row * nx), gy = static_cast<int>(row - plane * ny);
    const int gz = static_cast<int>(plane), P = fx.p;
    if (fx.zero_boundary && (gx == 0 || gx == fx.n[0] - 1 || gy == 0 || gy == fx.n[1] - 1 ||
                             (fx.n[2] > 1 && (gz == 0 || gz == fx.n[2] - 1)))) {
        rhs[g] = T(0);
        return;
    }
    if (!fx.spill) return;
    const int tx = min(gx / fx.tile[0], fx.nt[0] - 1), lx = gx - fx.tile[0] * tx;
    const int ty = min(gy / fx.tile[1], fx.nt[1] - 1), ly = gy - fx.tile[1] * ty;
    const int tz = min(gz / fx.tile[2], fx.nt[2] - 1), lz = gz - fx.tile[2] * tz;
    const bool sx = lx < P && tx > 0, sy = ly < P && ty > 0, sz = lz < P && tz > 0;
    if (!(sx || sy || sz)) return;
    double sum = 0;
#pragma unroll
    for (int d = 1; d < 8; ++d) {
        const int dx = d & 1, dy = (d >> 1) & 1, dz = d >> 2;
        if ((dx && !sx) || (dy && !sy) || (dz && !sz)) continue;
        sum += static_cast<double>(
            fx.spill[fx.off[d] + (dx ? tx * P + lx : gx) +
                     static_cast<long>(fx.ext[0][dx]) *
                         ((dy ? ty * P + ly : gy) + static_cast<long>(fx.ext[1][dy]) * (dz ? tz * P + lz : gz))]);
    }
    rhs[g] += static_cast<T>(sum);
}

// the fix-ups of two one-launch passes in one launch: blocks [0, half) the first, the rest
// the second
template <typename T>
__global__ __launch_bounds__(64 * kFixupRows) void k_rhs_fixup_pair(T* __restrict__ a, rhs_fixup<T> fa,
                                                                    T* __restrict__ b, rhs_fixup<T> fb, unsigned half) {
    if (blockIdx.x < half)
        rhs_fixup_block<T>(a, fa, blockIdx.x);
    else
        rhs_fixup_block<T>(b, fb, blockIdx.x - half);
}

// the end of a one-launch element loop (spill layout in q): its fix-up described for the
// caller (prm.defer), or launched now
template <typename T>
hipError_t finish_one(const rhs_params<T>& prm, const rhs_params<T>& q, T* rhs, int p, const int tile[3],
                      const int nt[3], const int n[3], hipStream_t s) {
    rhs_fixup<T> fx;
    defer_fixup(fx, q, p, tile, nt, n);
    if (prm.defer) {
        *prm.defer = fx;
        return hipSuccess;
    }
    return launch_rhs_fixup<T>(rhs, fx, s);
}

// The spill arrays of n[d] DOFs in nt[d] tiles per direction: array delta (1..7) has
// extent n[d] in the directions with delta_d = 0 and nt[d] P in the others, at off[delta];
// returns the total.
template <int P>
long spill_layout(const int n[3], const int nt[3], long off[8], int ext[3][2]) {
    for (int d = 0; d < 3; ++d) {
        ext[d][0] = n[d];
        ext[d][1] = nt[d] * P;
    }
    long total = 0;
    off[0] = 0;
    for (int delta = 1; delta < 8; ++delta) {
        off[delta] = total;
        total += static_cast<long>(ext[0][delta & 1]) * ext[1][(delta >> 1) & 1] * ext[2][delta >> 2];
    }
    return total;
}

// One launch over all tiles (variants 0, 1 and 2), then the spill fix-up over the DOFs.
template <typename T, int P, bool KF, int FM, int VAR>
hipError_t rhs3_one(const T* up, T* rhs, const dev_tables<T>* d, const rhs_params<T>& prm, hipStream_t s) {
    using TL = tile<3, P>;
    static_assert(VAR <= 2, "the other variants have no one-launch form here");
    const int ntx = (d[0].elements + TL::X - 1) / TL::X;
    const int nty = (d[1].elements + TL::Y - 1) / TL::Y;
    const int ntz = (d[2].elements + TL::Z - 1) / TL::Z;
    const long tiles = static_cast<long>(ntx) * nty * ntz;
    if (tiles == 0) return hipSuccess;
    if (!prm.spill) return hipErrorInvalidValue;
    // the spill arrays (sized by rhs_spill_slots for dofs = elements + P)
    rhs_params<T> q = prm;
    const int n[3] = {d[0].dofs, d[1].dofs, d[2].dofs}, nt[3] = {ntx, nty, ntz};
    for (int i = 0; i < 3; ++i)
        if (n[i] != d[i].elements + P) return hipErrorInvalidValue;
    spill_layout<P>(n, nt, q.spill_off, q.spill_ext);
    hipLaunchKernelGGL((k_rhs3<T, P, TL::X, TL::Y, TL::Z, KF, FM, VAR, true>), dim3(tiles),
                       dim3(TL::X * TL::Y * TL::Z), 0, s, up, rhs, d[0], d[1], d[2], q, 0, ntx, nty);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const int tl[3] = {TL::X, TL::Y, TL::Z};
    return finish_one(prm, q, rhs, P, tl, nt, n, s);
}

// Variant 4 in one launch: the marching kernel (adsg_rhs_march.hip) on its own tiles, then
// the spill fix-up over the DOFs.
template <typename T, int P>
hipError_t rhs3_march(const T* up, T* rhs, const dev_tables<T>* d, const rhs_params<T>& prm, const int tl[3],
                      const int nt[3], hipStream_t s) {
    if (d[0].elements <= 0 || d[1].elements <= 0 || d[2].elements <= 0) return hipSuccess;
    if (!prm.spill) return hipErrorInvalidValue;
    rhs_params<T> q = prm;
    const int n[3] = {d[0].dofs, d[1].dofs, d[2].dofs};
    for (int i = 0; i < 3; ++i)
        if (n[i] != d[i].elements + P) return hipErrorInvalidValue;
    spill_layout<P>(n, nt, q.spill_off, q.spill_ext);
    const hipError_t e = launch_rhs3_march<T>(P, up, rhs, d, q, tl, nt, s);
    if (e != hipSuccess) return e;
    return finish_one(prm, q, rhs, P, tl, nt, n, s);
}

// the largest spill total of the marching kernel's tiles over its precisions and forms
template <int P>
long rhs3_march_slots(const int elements[3]) {
    const int n[3] = {elements[0] + P, elements[1] + P, elements[2] + P};
    long most = 0;
    for (int k = 0; k < 4; ++k) {
        int tl[3], nt[3], ext[3][2];
        long off[8];
        rhs3_march_tiles(P, k & 1 ? 8 : 4, (k & 2) != 0, elements, tl, nt);
        most = std::max(most, spill_layout<P>(n, nt, off, ext));
    }
    return most;
}

// spill values of one launch of variants 0 to 2 (dofs = elements + P)
template <int P>
long rhs3_one_slots(const int elements[3]) {
    using TL = tile<3, P>;
    const int n[3] = {elements[0] + P, elements[1] + P, elements[2] + P};
    const int nt[3] = {(elements[0] + TL::X - 1) / TL::X, (elements[1] + TL::Y - 1) / TL::Y,
                       (elements[2] + TL::Z - 1) / TL::Z};
    long off[8];
    int ext[3][2];
    return spill_layout<P>(n, nt, off, ext);
}

// the 2D spill arrays: array delta (1..3) has extent n[d] in the directions with delta_d = 0
// and nt[d] P in the others; returns the total (off, ext as rhs_params holds them)
long spill_layout2(int p, const int n[2], const int nt[2], long off[8], int ext[3][2]) {
    for (int d = 0; d < 2; ++d) {
        ext[d][0] = n[d];
        ext[d][1] = nt[d] * p;
    }
    ext[2][0] = ext[2][1] = 1;
    long total = 0;
    for (int k = 0; k < 8; ++k) off[k] = 0;
    for (int delta = 1; delta < 4; ++delta) {
        off[delta] = total;
        total += static_cast<long>(ext[0][delta & 1]) * ext[1][delta >> 1];
    }
    return total;
}

// the 3D k-field gradient on the tiles of tile<3, P>: one launch over all tiles and the
// fix-up when prm has a spill buffer (owned entries added), else one launch per colour
template <typename T, int P>
hipError_t kgrad3(const T* u, const T* w, T* out, const dev_tables<T>* d, const rhs_params<T>& prm, hipStream_t s) {
    using TL = tile<3, P>;
    constexpr int NT = TL::X * TL::Y * TL::Z;
    const int ntx = (d[0].elements + TL::X - 1) / TL::X;
    const int nty = (d[1].elements + TL::Y - 1) / TL::Y;
    const int ntz = (d[2].elements + TL::Z - 1) / TL::Z;
    if (ntx <= 0 || nty <= 0 || ntz <= 0) return hipSuccess;
    const int n[3] = {d[0].dofs, d[1].dofs, d[2].dofs}, nt[3] = {ntx, nty, ntz};
    for (int i = 0; i < 3; ++i)
        if (n[i] != d[i].elements + P) return hipErrorInvalidValue;
    rhs_params<T> q = prm;
    q.kfield = w;  // staged as the k block
    q.store = false;
    q.defer = nullptr;
    if (prm.spill) {
        spill_layout<P>(n, nt, q.spill_off, q.spill_ext);
        const long tiles = static_cast<long>(ntx) * nty * ntz;
        hipLaunchKernelGGL((k_kgrad3<T, P, TL::X, TL::Y, TL::Z, true>), dim3(tiles), dim3(NT), 0, s, u, out, d[0],
                           d[1], d[2], q, 0, ntx, nty);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        const int tl[3] = {TL::X, TL::Y, TL::Z};
        return finish_one(q, q, out, P, tl, nt, n, s);
    }
    for (int c = 0; c < 8; ++c) {
        const int nx2 = (ntx - (c & 1) + 1) / 2, ny2 = (nty - ((c >> 1) & 1) + 1) / 2;
        const int nz2 = (ntz - ((c >> 2) & 1) + 1) / 2;
        const long tiles = static_cast<long>(nx2) * ny2 * nz2;
        if (tiles == 0) continue;
        hipLaunchKernelGGL((k_kgrad3<T, P, TL::X, TL::Y, TL::Z, false>), dim3(tiles), dim3(NT), 0, s, u, out, d[0],
                           d[1], d[2], q, c, nx2, ny2);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// the 2D k-field gradient: one launch over all tiles and the fix-up when prm has a spill
// buffer (prm.store false: the owned entries are added), else one launch per parity colour
template <typename T, int P>
hipError_t kgrad2(const T* u, const T* w, T* out, const dev_tables<T>* d, const rhs_params<T>& prm, hipStream_t s) {
    using TL = tile<2, P>;
    const int ntx = (d[0].elements + TL::X - 1) / TL::X, nty = (d[1].elements + TL::Y - 1) / TL::Y;
    if (ntx <= 0 || nty <= 0) return hipSuccess;
    if (d[0].dofs != d[0].elements + P || d[1].dofs != d[1].elements + P) return hipErrorInvalidValue;
    if (prm.spill) {
        rhs_params<T> q = prm;
        q.store = false;
        q.defer = nullptr;
        const int n[2] = {d[0].dofs, d[1].dofs}, nt[2] = {ntx, nty};
        spill_layout2(P, n, nt, q.spill_off, q.spill_ext);
        hipLaunchKernelGGL((k_kgrad2<T, P, TL::X, TL::Y, true>), dim3(ntx * nty), dim3(TL::X * TL::Y), 0, s, u, w, out,
                           d[0], d[1], q, 0, ntx);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        const int tl[3] = {TL::X, TL::Y, 1}, nt3[3] = {ntx, nty, 1}, n3[3] = {n[0], n[1], 1};
        return finish_one(q, q, out, P, tl, nt3, n3, s);
    }
    for (int c = 0; c < 4; ++c) {
        const int nx2 = (ntx - (c & 1) + 1) / 2, ny2 = (nty - ((c >> 1) & 1) + 1) / 2;
        if (nx2 * ny2 == 0) continue;
        hipLaunchKernelGGL((k_kgrad2<T, P, TL::X, TL::Y, false>), dim3(nx2 * ny2), dim3(TL::X * TL::Y), 0, s, u, w,
                           out, d[0], d[1], prm, c, nx2);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

template <typename T, int P, int FM, int VAR>
hipError_t rhs3_forms(const T* up, T* rhs, const dev_tables<T>* d, const rhs_params<T>& prm,
                      hipStream_t s) {
    const bool kf = prm.kfield != nullptr;
    if (kf) return rhs3_colours<T, P, true, FM, VAR>(up, rhs, d, prm, s);
    return rhs3_colours<T, P, false, FM, VAR>(up, rhs, d, prm, s);
}

template <typename T, int P, int VAR>
hipError_t rhs3_fields(const T* up, T* rhs, const dev_tables<T>* d, const rhs_params<T>& prm,
                       bool one, hipStream_t s) {
    // one launch (forms without a k field; checked by the caller)
    if constexpr (VAR <= 2) {
        if (one) {
            if (prm.reaction != T(0)) return rhs3_one<T, P, false, 1, VAR>(up, rhs, d, prm, s);
            if (prm.mass == T(0)) return rhs3_one<T, P, false, 2, VAR>(up, rhs, d, prm, s);
            return rhs3_one<T, P, false, 0, VAR>(up, rhs, d, prm, s);
        }
    }
    if (prm.reaction != T(0)) return rhs3_forms<T, P, 1, VAR>(up, rhs, d, prm, s);
    if (prm.mass == T(0) && !prm.kfield)
        return rhs3_colours<T, P, false, 2, VAR>(up, rhs, d, prm, s);
    return rhs3_forms<T, P, 0, VAR>(up, rhs, d, prm, s);
}

template <typename T, int P>
hipError_t rhs_fields(int dim, const T* up, T* rhs, const dev_tables<T>* d,
                      const rhs_params<T>& prm_in, int code, hipStream_t s) {
    rhs_params<T> prm = prm_in;
    const bool kf = prm.kfield != nullptr;
    // bits 4..7: the shape of variant 5; bit 8: one launch; bit 9: overwrite
    int variant = code & 15;
    if (dim == 3 && variant == 5 && !rhs3_col_supported<T>(P, prm)) variant = P == 3 ? 2 : 1;
    // element columns on the matrix cores where the form allows, else the degree's default
    // per-element variant
    bool one = dim == 3 && (code & kRhsOneLaunch) != 0 && prm.spill && variant != 3 && variant != 5;
    // 3D in one launch: the marching kernel for variant 4 and, where it is faster, for forms with a
    // k field, which the per-element kernels take in colour launches only (70 x 50 x 61, p = 2,
    // FP64: 34 us against 154 us in eight launches and a fill)
    bool march = one && (kf ? rhs3_march_kfield<T>(P) : variant == 4);
    int tl[3], nt[3];
    if (march) {
        const int el[3] = {d[0].elements, d[1].elements, d[2].elements};
        const double cost = rhs3_march_tiles(P, sizeof(T), kf, el, tl, nt);
        march = rhs3_march_fits(sizeof(T), d[0].dofs, d[1].dofs, nt) &&
                (!kf || rhs3_march_pays(P, sizeof(T), true, el, cost));
    }
    one = one && (!kf || march);
    const bool marched = dim == 2 || march;
    if (one && variant == 4 && !marched) variant = P == 3 ? 2 : 1;
    const long n = static_cast<long>(d[0].dofs) * d[1].dofs * (dim == 3 ? d[2].dofs : 1);
    bool overwrite = (code & kRhsOverwrite) != 0;
    if (prm.start && !marched) {  // the marching kernels add it as they write
        const hipError_t e = launch_scale<T>(rhs, prm.start, n, prm.start_scale, s);
        if (e != hipSuccess) return e;
        prm.start = nullptr;
        overwrite = false;
    }
    // overwrite: the one launch's owners and the 2D strips store; the colour launches add into
    // a zero fill
    prm.store = overwrite && !prm.start && (one || dim == 2);
    if (overwrite && !one && dim != 2) {
        const hipError_t e = launch_fill<T>(rhs, n, T(0), s);
        if (e != hipSuccess) return e;
    }
    if (dim == 3) {
        if (marched) return rhs3_march<T, P>(up, rhs, d, prm, tl, nt, s);
        if (variant == 5) return launch_rhs3_col<T>(P, up, rhs, d, prm, (code >> 4) & 15, s);
        if (variant == 1) return rhs3_fields<T, P, 1>(up, rhs, d, prm, one, s);
        if (variant == 2) return rhs3_fields<T, P, 2>(up, rhs, d, prm, one, s);
        if (variant == 3) return rhs3_fields<T, P, 3>(up, rhs, d, prm, one, s);
        if (variant == 4) return rhs3_fields<T, P, 4>(up, rhs, d, prm, one, s);
        return rhs3_fields<T, P, 0>(up, rhs, d, prm, one, s);
    }
    return launch_rhs2_march<T>(P, up, rhs, d, prm, s);
}

}  // namespace

template <typename T>
hipError_t launch_rhs(int dim, int p, const T* u_prev, T* rhs, const dev_tables<T>* dirs,
                      const rhs_params<T>& prm, int variant, hipStream_t s) {
    switch (p) {
        case 1:
            return rhs_fields<T, 1>(dim, u_prev, rhs, dirs, prm, variant, s);
        case 2:
            return rhs_fields<T, 2>(dim, u_prev, rhs, dirs, prm, variant, s);
        case 3:
            return rhs_fields<T, 3>(dim, u_prev, rhs, dirs, prm, variant, s);
        default:
            return hipErrorInvalidValue;
    }
}

// the 2D adjoint pair (k_adjoint2): out_r := the element loop of prm_r for w (stored: the
// start value of out_r is unused), out_k += the k-field gradient of u and w; spill_r and
// spill_k: two spill arrays of rhs_spill_slots(2, p, ...) values
template <typename T, int P>
hipError_t adjoint2(const T* w, const T* u, T* out_r, T* out_k, const dev_tables<T>* d, const rhs_params<T>& prm_r,
                    const rhs_params<T>& prm_k, T* spill_r, T* spill_k, hipStream_t s) {
    using TL = tile<2, P>;
    const int ntx = (d[0].elements + TL::X - 1) / TL::X, nty = (d[1].elements + TL::Y - 1) / TL::Y;
    const int tiles = ntx * nty;
    if (tiles <= 0) return hipSuccess;
    if (d[0].dofs != d[0].elements + P || d[1].dofs != d[1].elements + P || !spill_r || !spill_k)
        return hipErrorInvalidValue;
    const int n[2] = {d[0].dofs, d[1].dofs}, nt[2] = {ntx, nty};
    rhs_params<T> qr = prm_r, qk = prm_k;
    qr.spill = spill_r;
    qr.store = true;
    qr.defer = nullptr;
    qk.spill = spill_k;
    qk.store = false;
    qk.defer = nullptr;
    spill_layout2(P, n, nt, qr.spill_off, qr.spill_ext);
    spill_layout2(P, n, nt, qk.spill_off, qk.spill_ext);
    hipLaunchKernelGGL((k_adjoint2<T, P, TL::X, TL::Y>), dim3(2 * tiles), dim3(TL::X * TL::Y), 0, s, w, u, out_r, out_k,
                       d[0], d[1], qr, qk, ntx, tiles);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const int tl[3] = {TL::X, TL::Y, 1}, nt3[3] = {ntx, nty, 1}, n3[3] = {n[0], n[1], 1};
    rhs_fixup<T> fr, fk;
    defer_fixup(fr, qr, P, tl, nt3, n3);
    defer_fixup(fk, qk, P, tl, nt3, n3);
    const unsigned half = static_cast<unsigned>((n[1] + kFixupRows - 1) / kFixupRows);
    hipLaunchKernelGGL((k_rhs_fixup_pair<T>), dim3(2 * half), dim3(64 * kFixupRows), 0, s, out_r, fr, out_k, fk, half);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_adjoint2(int p, const T* w, const T* u, T* out_r, T* out_k, const dev_tables<T>* dirs,
                           const rhs_params<T>& prm_r, const rhs_params<T>& prm_k, T* spill_r, T* spill_k,
                           hipStream_t s) {
    switch (p) {
        case 1:
            return adjoint2<T, 1>(w, u, out_r, out_k, dirs, prm_r, prm_k, spill_r, spill_k, s);
        case 2:
            return adjoint2<T, 2>(w, u, out_r, out_k, dirs, prm_r, prm_k, spill_r, spill_k, s);
        case 3:
            return adjoint2<T, 3>(w, u, out_r, out_k, dirs, prm_r, prm_k, spill_r, spill_k, s);
        default:
            return hipErrorInvalidValue;
    }
}

template <typename T>
hipError_t launch_kgrad(int dim, int p, const T* u, const T* w, T* out, const dev_tables<T>* dirs,
                        const rhs_params<T>& prm, hipStream_t s) {
    if (dim != 2 && dim != 3) return hipErrorInvalidValue;
    switch (p) {
        case 1:
            return dim == 2 ? kgrad2<T, 1>(u, w, out, dirs, prm, s) : kgrad3<T, 1>(u, w, out, dirs, prm, s);
        case 2:
            return dim == 2 ? kgrad2<T, 2>(u, w, out, dirs, prm, s) : kgrad3<T, 2>(u, w, out, dirs, prm, s);
        case 3:
            return dim == 2 ? kgrad2<T, 3>(u, w, out, dirs, prm, s) : kgrad3<T, 3>(u, w, out, dirs, prm, s);
        default:
            return hipErrorInvalidValue;
    }
}

long rhs2_spill_layout(int p, int tx, int ty, const int elements[2], long off[8], int ext[3][2]) {
    const int n[2] = {elements[0] + p, elements[1] + p};
    const int nt[2] = {(elements[0] + tx - 1) / tx, (elements[1] + ty - 1) / ty};
    return spill_layout2(p, n, nt, off, ext);
}

template <typename T>
hipError_t launch_rhs_fixup(T* rhs, const rhs_fixup<T>& fx, hipStream_t s) {
    if (!fx.pending()) return hipSuccess;
    const long rows = static_cast<long>(fx.n[1]) * fx.n[2];
    if (rows <= 0 || fx.n[0] <= 0) return hipSuccess;
    const long N = rows * fx.n[0];
    if (fx.n[0] < kFixupRowLength && rows >= kFixupManyRows && N < (1L << 31)) {
        hipLaunchKernelGGL((k_rhs_fixup_dofs<T>), dim3(static_cast<unsigned>((N + 255) / 256)), dim3(256), 0, s, rhs,
                           fx, static_cast<unsigned>(N));
        return hipGetLastError();
    }
    const unsigned blocks = static_cast<unsigned>((rows + kFixupRows - 1) / kFixupRows);
    for (unsigned b = 0; b < blocks; b += kFixupBlocks)
        hipLaunchKernelGGL((k_rhs_fixup<T>), dim3(std::min(blocks - b, kFixupBlocks)), dim3(64 * kFixupRows), 0, s, rhs,
                           fx, b);
    return hipGetLastError();
}

long rhs_spill_slots(int dim, int p, const int elements[3]) {
    if (dim == 2) {
        long off[8];
        int ext[3][2];
        return p >= 1 && p <= 3 ? rhs2_spill_layout(p, 16, 16, elements, off, ext) : 0;
    }
    switch (p) {
        case 1:
            return std::max(rhs3_one_slots<1>(elements), rhs3_march_slots<1>(elements));
        case 2:
            return std::max(rhs3_one_slots<2>(elements), rhs3_march_slots<2>(elements));
        case 3:
            return std::max(rhs3_one_slots<3>(elements), rhs3_march_slots<3>(elements));
        default:
            return 0;
    }
}

// Modelled times, us: the march takes its cost in planes times kPlane; the per-element kernels in
// one launch a time per tile (kStart: the difference of what neither grows with), the colour launches
// at least kLaunch each, more with many tiles. A march pads x to 31 / 19 / 16 elements and y to 4, the
// tiles x and y to 8, so on thin meshes and those just over a tile the element count alone chose
// wrongly. Fitted to the step times of 39 meshes per degree and
// precision (32^3 to 160^3, 1 to 39 or 130 to 300 elements along x, 1 to 17 along y or z; p = 3 FP64 68):
// the kernel chosen is 0.02 to 0.65 % slower than the faster one on average, 8 % at most (by
// element count 5 % in FP64 for p = 2 and 3, 82 % at most; with a k field always marching 3 %, 53 %
// at most). Examples, march against per-element: 128^3 FP64 p = 1 96 / 101, p = 2 176 / 229, p = 3
// 389 / 759; 8 x 256 x 256 p = 2 FP64 119 / 92; 17 x 140 x 140 p = 2 FP64 68 / 82; 5 x 300 x 300
// p = 3 FP64 335 / 256, with a k field 433 against 314 in colours. One element along x or y takes the
// colour launches of p = 3 half as long again as two.
bool rhs3_march_pays(int p, int bytes, bool kfield, const int elements[3], double cost) {
    if (p < 1 || p > 3) return false;
    const int f32 = bytes == 4;
    const int te[3] = {8, 8, p == 3 ? 3 : 4};  // tile<3, p>
    double tiles = 1, launches = 1;
    for (int d = 0; d < 3; ++d) {
        const int n = (elements[d] + te[d] - 1) / te[d];
        tiles *= n;
        if (n > 1) launches *= 2;
    }
    if (!kfield) {
        static const double kPlane[2][4] = {{0, 1.0, 2.2, 3.8}, {0, 0.71, 1.5, 2.4}};
        static const double kTile[2][4] = {{0, 5.4e-3, 20e-3, 57e-3}, {0, 3.3e-3, 11e-3, 32e-3}};
        static const double kStart[2][4] = {{0, -1.7, -8.2, -25}, {0, -0.36, -5.2, -13}};
        return kPlane[f32][p] * cost + kStart[f32][p] < kTile[f32][p] * tiles;
    }
    if (p == 3 && (elements[0] == 1 || elements[1] == 1)) return true;
    static const double kPlane[2][4] = {{0, 1.1, 1.2, 3.6}, {0, 1.0, 1.7, 3.6}};
    static const double kLaunch[2][4] = {{0, 4.6, 17, 30}, {0, 4.5, 9.5, 30}};
    static const double kOverlap[2][4] = {{0, 2.3, 8.5, 20}, {0, 2.25, 4.75, 20}};
    static const double kTile[2][4] = {{0, 6e-3, 21e-3, 64e-3}, {0, 6e-3, 12.5e-3, 64e-3}};
    return kPlane[f32][p] * cost <
           launches * std::max(kLaunch[f32][p], kOverlap[f32][p] + kTile[f32][p] * tiles / launches);
}

void rhs2_batch_tiles(int elements_x, int elements_y, int ntx2[4], int count[4]) {
    const int ntx = (elements_x + 7) / 8, nty = (elements_y + 7) / 8;
    for (int c = 0; c < 4; ++c) {
        const int cx = c & 1, cy = (c >> 1) & 1;
        ntx2[c] = (ntx - cx + 1) / 2;
        count[c] = ntx2[c] * ((nty - cy + 1) / 2);
    }
}

template <typename T>
hipError_t launch_rhs2_batch(int p, const rhs2_item<T>* items, int nitems, int colour, int blocks, hipStream_t s) {
    if (blocks <= 0 || nitems <= 0) return hipSuccess;
    if (p == 1)
        hipLaunchKernelGGL((k_rhs2_batch<T, 1, 8>), dim3(blocks), dim3(64), 0, s, items, nitems, colour);
    else if (p == 2)
        hipLaunchKernelGGL((k_rhs2_batch<T, 2, 8>), dim3(blocks), dim3(64), 0, s, items, nitems, colour);
    else if (p == 3)
        hipLaunchKernelGGL((k_rhs2_batch<T, 3, 8>), dim3(blocks), dim3(64), 0, s, items, nitems, colour);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

template hipError_t launch_kgrad<double>(int, int, const double*, const double*, double*, const dev_tables<double>*,
                                         const rhs_params<double>&, hipStream_t);
template hipError_t launch_adjoint2<double>(int, const double*, const double*, double*, double*,
                                            const dev_tables<double>*, const rhs_params<double>&,
                                            const rhs_params<double>&, double*, double*, hipStream_t);
template hipError_t launch_rhs_fixup<double>(double*, const rhs_fixup<double>&, hipStream_t);
template hipError_t launch_rhs_fixup<float>(float*, const rhs_fixup<float>&, hipStream_t);
template hipError_t launch_rhs2_batch<double>(int, const rhs2_item<double>*, int, int, int, hipStream_t);
template hipError_t launch_rhs2_batch<float>(int, const rhs2_item<float>*, int, int, int, hipStream_t);
template hipError_t launch_rhs<double>(int, int, const double*, double*, const dev_tables<double>*,
                                       const rhs_params<double>&, int, hipStream_t);
template hipError_t launch_rhs<float>(int, int, const float*, float*, const dev_tables<float>*,
                                      const rhs_params<float>&, int, hipStream_t);

}  // namespace adsg

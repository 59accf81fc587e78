// HIP kernels of the vorticity-equation step and the tracer loop (gfx950).
//
// Device data layout (one GPU holds the whole periodic box, cubic N^3):
//   spectral plane  [ky][kz][kx],  kx = 0 .. N/2-1 stored (NXH = N/2)
//   real plane      [y][z][x],     x  = 0 .. N-1
// A vector field is 3 (or 6, 9) planes plane_size(N) complex values apart;
// within a plane, ky (or y) rows are row_stride(N) = N*NXH + BFPSH_PAD_Y
// complex apart (common.hpp), and a real row (y, z) occupies the bytes of
// the spectral row (ky = y, kz = z).  The kx = N/2 plane of the reference's
// half spectrum is not stored: it lies outside the dealiasing sphere
// (kx^2 >= (N/2)^2 > kM^2), the reference's io_checkpoint read zeroes it
// (low_pass, bfps/cpp/kspace.cpp:235-253) and the time step never writes it
// (bfps/cpp/vorticity_equation.cpp:372), so it is identically zero.
//
// The step's inverse transforms run y pass -> z pass -> x (c2r) pass and its
// forward transforms x (r2c) -> z -> y, so that the last forward pass of one
// Runge-Kutta stage and the first inverse pass of the next are both along y
// and run in one kernel (k_y_update).  Standalone fields run z -> y -> x and
// x -> z -> y.  The real-space array comes out as [y][z][x]; the x passes
// work on pairs of rows (z, z+1) packed as the real and imaginary parts of
// one complex sequence.
//
// Band table.  Outside the dealiasing sphere k^2 <= kM^2 the velocity is zero
// and so is the vorticity (unless a caller put unprojected data).  Where the
// pencil along y at (kx, kz) lies outside the sphere altogether (21 % of the
// pencils with the smooth filter, 65 % under the two-thirds rule) the step
// neither transforms nor moves it: zl[kx] is the largest |kz| of column kx
// that reaches the sphere (-1: none; not increasing with kx), zl[N / 2] the
// largest such kx.  Every kernel of the step reads the same table, so what
// one leaves unwritten no other reads.
#pragma once
#include "fft.hpp"

#ifndef BFPSH_TILE_BYTES
#define BFPSH_TILE_BYTES 128
#endif
// LDS bytes a tile of the plain strided pass may take (B columns x N
// complex values; gfx950 has 160 KB of LDS per CU)
#ifndef BFPSH_TILE_LDS
#define BFPSH_TILE_LDS 131072
#endif
// register-resident x pass (k_rows_cross_w): minimum waves per SIMD and
// LDS padding (one slot every 2^BFPSH_RW_PAD rows); measured at 512^3 FP32,
// 3 waves with padding every 16 rows beat 2 waves with padding every 8
#ifndef BFPSH_RW_WAVES
#define BFPSH_RW_WAVES 3
#endif
#ifndef BFPSH_RW_PAD
#define BFPSH_RW_PAD 4
#endif

namespace bfpsh {

// ------------------------------------------------------------ configuration
template <typename T, int N>
struct Cfg {
    static constexpr int NXH = N / 2;
    static constexpr int RMAX = 16;  // radix cap of the LDS-tile FFT (row passes)
    // plain strided passes: register-resident FFT, E complex values per
    // thread (all radices divide E)
    static constexpr int ereg() {
        if (N % 3 == 0) return 12;
        if (N <= 16) return N;
        if (sizeof(T) == 4 && (N == 128 || N == 256 || N == 1024)) return 16;
        return 8;
    }
    static constexpr int E = ereg();
    // columns per strided tile: BFPSH_TILE_BYTES-byte row segments (default
    // 128) in at most lds bytes of LDS
    static constexpr int bcap(int lds) {
        int b = int(BFPSH_TILE_BYTES / sizeof(C2<T>));
        const int lim = int(lds / (N * sizeof(C2<T>)));
        if (b > lim) b = lim;
        if (b > NXH) b = NXH;
        while (NXH % b) b /= 2;
        return b;
    }
    // plain strided pass (k_pass): up to BFPSH_TILE_LDS bytes, which only
    // widens the 1024^3 tiles (FP32 8 -> 16 columns: one y pass over a plane
    // 2.97 -> 2.46 ms); the fused first and last passes keep 64 KB tiles
    // (their three components in registers need the smaller workgroups)
    static constexpr int B = bcap(BFPSH_TILE_LDS);
    static constexpr int BF = bcap(65536);
    // fused y passes (Biot-Savart, update): three components stay in
    // registers.  Small boxes run one short wave of workgroups, whose time is
    // the code each one walks through once: fewer values per thread (FP32
    // first stage at 16^3, 2 / 4 / 16 values: 11.1 / 13.7 / 22.5 us; 64^3,
    // 4 / 8: 17.6 / 22.1 us; 256^3, 8 / 16: 218 / 239 us)
    static constexpr int efused() {
        if (N % 3 == 0) return 6;
        if (N <= 32) return 2;
        if (N == 64) return 4;
        if (N <= 256) return 8;
        return E;
    }
    // half the columns when the threads would exceed 512, to keep the
    // Biot-Savart pass within a 256-VGPR budget
    static constexpr int E_BS = efused();
    static constexpr int B_BS = ((N / E_BS) * BF > 512 && BF > 1) ? BF / 2 : BF;
    static constexpr int NT_BS = (N / E_BS) * B_BS;
    // last forward pass with the update epilogue (3 components in registers)
    static constexpr int E_Y3 = efused();
    static constexpr int B_Y3 = BF;
    static constexpr int NT_Y3 = (N / E_Y3) * B_Y3;
    // elements per thread of the plain strided pass (measured at 512^3 FP32:
    // 16 elements x 512 threads beat 8 x 1024)
#ifndef BFPSH_E_PASS
#define BFPSH_E_PASS 16
#endif
    static constexpr int pick_e(int e, int b) { return (e > 0 && N % e == 0 && (N / e) * b <= 1024) ? e : E; }
    static constexpr int E_PASS = pick_e(sizeof(T) == 4 && N == 512 ? BFPSH_E_PASS : 0, B);
    static constexpr int RP = (N * int(sizeof(C2<T>)) >= 8192) ? 1 : 2;  // row pairs per row block
    // threads of the LDS-tile row passes (1024: two blocks of 512 per CU,
    // four waves per SIMD, instead of two blocks of 256)
    static constexpr int NT_ROW = N >= 1024 ? 512 : (N >= 256 ? 256 : (N >= 64 ? 128 : 64));
    // LDS row stride of the LDS-tile cross-product pass (6 RP components per
    // row): odd, spreading strided lanes over the banks, unless that slot
    // costs a resident workgroup per CU (1024^3 FP32: three 48 KB
    // workgroups instead of two of 56 KB, 14.4 -> 12.0 ms per launch)
    static constexpr int ls_row() {
        const long c = 6 * RP, lds = 160 * 1024, row = long(N) * long(sizeof(C2<T>));
        return lds / (row * c) > lds / (row * (c + 1)) ? int(c) : int(c + 1);
    }
    static constexpr int LS_ROW = ls_row();
    static_assert((N / E_PASS) * B <= 1024 && (N / E_Y3) * B_Y3 <= 1024, "tile threads");
};

// offsets of row (y, z), row = y N + z, of a plane: complex values of a
// spectral row and reals of a real row (the same bytes)
template <int N> BFPSH_DEV size_t crow(size_t row) { return (row / N) * row_stride(N) + (row % N) * (N / 2); }
template <int N> BFPSH_DEV size_t rrow(size_t row) { return (row / N) * 2 * row_stride(N) + (row % N) * N; }

// Element at a byte offset of 32 bits from a pointer that is uniform over the
// workgroup: the pointer stays in scalar registers and one vector register of
// offset serves every row g + G m (the G m rows are part of the pointer) and
// every plane.  A thread's own offset (row g, column) stays below 2^31 bytes.
template <typename T> BFPSH_DEV C2<T>& at_off(C2<T>* p, uint32_t off) {
    return *reinterpret_cast<C2<T>*>(reinterpret_cast<char*>(p) + off);
}
template <typename T> BFPSH_DEV const C2<T>& at_off(const C2<T>* p, uint32_t off) {
    return *reinterpret_cast<const C2<T>*>(reinterpret_cast<const char*>(p) + off);
}

// ------------------------------------------------------------ parameters
struct Geom {
    int n;
    double dkx, dky, dkz;
    double kM2;
    int smooth;  // 1: smooth filter exp(-36 (k^2/kM^2)^18), 0: two-thirds low pass
};
struct StepParams {
    double nu, dt, famp, fk0, fk1;
    int forcing;  // 0 none, 1 linear, 2 Kolmogorov, 3 fixed energy-injection rate
    int fmode;
    const double* famp_dev;  // forcing 3: band amplitudes of the 3 stages (device)
};

BFPSH_DEV double kwave(int i, int n, double dk) { return (i <= n / 2 ? i : i - n) * dk; }

// a -= k (k . a) / k^2 (force_divfree, bfps/cpp/kspace.cpp:487-519), ik2 = 1 / k^2
template <typename T>
BFPSH_DEV void divfree(C2<T> (&a)[3], double kx, double ky, double kz, double ik2) {
    const T t0 = T((kx * a[0].x + ky * a[1].x + kz * a[2].x) * ik2);
    const T t1 = T((kx * a[0].y + ky * a[1].y + kz * a[2].y) * ik2);
    a[0] = mk<T>(T(a[0].x - t0 * kx), T(a[0].y - t1 * kx));
    a[1] = mk<T>(T(a[1].x - t0 * ky), T(a[1].y - t1 * ky));
    a[2] = mk<T>(T(a[2].x - t0 * kz), T(a[2].y - t1 * kz));
}

// Workgroups are dealt round-robin to the 8 XCDs (each with its own L2).
// Remap a 2D grid so that each XCD walks a contiguous range of logical blocks
// (x fastest): neighbouring x tiles, which share 128-byte lines when a tile
// row is 64 bytes, then run on the same XCD back to back.
BFPSH_DEV void xcd_tile(int& bx, int& by) {
    const unsigned gx = gridDim.x, total = gridDim.x * gridDim.y;
    unsigned p = blockIdx.x + blockIdx.y * gx;
    if (total % 8u == 0) p = (p % 8u) * (total / 8u) + p / 8u;
    bx = int(p % gx);
    by = int(p / gx);
}

// ------------------------------------------------------------ K1 + first inverse pass
// MODE 0: outputs u_hat (3), omega_hat (3)        [nonlinear term]
// MODE 1: outputs u_hat (3)                        [velocity in real space]
// MODE 2: outputs i k_j u_hat_i (9), k^2 < kM^2    [velocity gradient]
// u_hat = i k x omega_hat / k^2 for 0 < k^2 <= kM^2, else 0
// (compute_velocity, bfps/cpp/vorticity_equation.cpp:206-239;
// compute_gradient, bfps/cpp/field.cpp:1077-1097).
template <int MODE> struct BsOut { static constexpr int NF = MODE == 0 ? 6 : (MODE == 1 ? 3 : 9); };

// compute_velocity symmetrizes u_hat on the kx = 0 plane: its lower half
// (ky > N/2, or ky = 0 and kz > N/2) becomes the conjugated mirror of the
// upper half (field.cpp:900-978).  The c2r pass takes the real part of the
// kx = 0 sum, to which a mode and its conjugated mirror add the same, so the
// lower half may be left out and the upper half doubled: this factor of a
// kx = 0 mode, with no mirror to read.  (A z derivative at kz = N/2, whose
// mirror has the same kz, is no such pair: see MODE 2 below.)
template <typename T, int N> BFPSH_DEV T plane0_factor(int ky, int kz) {
    if (ky > N / 2 || (ky == 0 && kz > N / 2)) return T(0);
    if (ky == N / 2 || (ky == 0 && (kz == 0 || kz == N / 2))) return T(1);  // its own mirror, or none
    return T(2);
}

// Velocity component cu of the mode (kx, ky, kz) with vorticity a0, a1, a2,
// zero outside 0 < k^2 <= kM^2
template <typename T>
BFPSH_DEV C2<T> biot_savart(int cu, C2<T> a0, C2<T> a1, C2<T> a2, double kx, double ky, double kz, double k2,
                            double kM2) {
    C2<T> u = mk<T>(T(0), T(0));
    if (k2 <= kM2 && k2 > 0) {
        // one FP64 division per element and field, then products (within
        // an ulp of the quotients before the rounding to T)
        const double ik2 = 1.0 / k2;
        if (cu == 0) u = mk<T>(T(-(ky * a2.y - kz * a1.y) * ik2), T((ky * a2.x - kz * a1.x) * ik2));
        if (cu == 1) u = mk<T>(T(-(kz * a0.y - kx * a2.y) * ik2), T((kz * a0.x - kx * a2.x) * ik2));
        if (cu == 2) u = mk<T>(T(-(kx * a1.y - ky * a0.y) * ik2), T((kx * a1.x - ky * a0.x) * ik2));
    }
    return u;
}

// offset of row g, column kxi of a y pencil
template <typename T, int N> BFPSH_DEV uint32_t y_off(int g, int kxi) {
    return (uint32_t(g) * uint32_t(row_stride(N)) + uint32_t(kxi)) * uint32_t(sizeof(C2<T>));
}

// LDS tiles of the fused y passes: two (one barrier an exchange, nine
// transforms a workgroup) wherever two tiles take at most the 128 KB that
// leave the integrating-factor table its room
template <typename T, int N> constexpr int fused_bufs(int b) { return N * b * int(sizeof(C2<T>)) <= 65536 ? 2 : 1; }

// Fields of the column (kxi, kz) from its vorticity wr (element e at row
// F::in_row(grp, e)), inverse-transformed along y into o + f PS, f < NF.
template <typename T, int N, int MODE, class F, int E, int NBUF>
BFPSH_DEV void bs_inverse_y(C2<T> (&wr)[3][E], C2<T>* lds, int cur, const C2<T>* __restrict__ tw, C2<T>* o, int grp,
                            int b, int kxi, int kz, const Geom& g) {
    constexpr size_t PS = plane_size(N), GS = F::G * row_stride(N);
    o += size_t(kz) * (N / 2);
    constexpr int NF = BsOut<MODE>::NF;
    const double kx = kxi * g.dkx, kzv = kwave(kz, N, g.dkz);
    // Velocity-type fields in a runtime loop (register arrays indexed by
    // constants only), then the vorticity copies (MODE 0) as straight-line
    // code: a runtime select between wr[0..2] would turn into a pointer into
    // wr and force the array into scratch memory.
    constexpr int NU = MODE == 0 ? 3 : NF;
#pragma unroll 1
    for (int f = 0; f < NU; f++) {
        // an opaque copy of the group index: the per-element wavenumbers are
        // recomputed per output field instead of being held across the loop
        int gq = grp;
        asm volatile("" : "+v"(gq));
        // likewise the source values: products of them with the wavenumbers
        // would otherwise be hoisted (in FP64) out of the loop
#pragma unroll
        for (int e = 0; e < E; e++)
#pragma unroll
            for (int c = 0; c < 3; c++) asm volatile("" : "+v"(wr[c][e].x), "+v"(wr[c][e].y));
        C2<T> v[E];
#pragma unroll
        for (int e = 0; e < E; e++) {
            const int n = F::in_row(gq, e);
            const double kyv = kwave(n, N, g.dky);
            const double k2 = kx * kx + kyv * kyv + kzv * kzv;
            const int cu = MODE == 2 ? f % 3 : f;
            C2<T> u = biot_savart<T>(cu, wr[0][e], wr[1][e], wr[2][e], kx, kyv, kzv, k2, g.kM2);
            if (kxi == 0) {
                const T s = plane0_factor<T, N>(n, kz);
                u = mk<T>(u.x * s, u.y * s);
            }
            if (MODE == 2) {
                const int j = f / 3;
                const double kj = j == 0 ? kx : (j == 1 ? kyv : kzv);
                // i k_z of a kx = 0 mode at kz = N/2 and of its mirror, both
                // at +N/2: their sum has no real part, where doubling one
                // counts the part that the mirror cancels
                const bool cancels = kxi == 0 && j == 2 && kz == N / 2 && n > 0 && n < N / 2;
                v[e] = k2 < g.kM2 && !cancels ? mk<T>(T(-kj * u.y), T(kj * u.x)) : mk<T>(T(0), T(0));
            } else {
                v[e] = u;
            }
        }
        F::template run<NBUF, true>(v, lds, tw, gq, b, cur);
        C2<T>* of = o + size_t(f) * PS;
#pragma unroll
        for (int e = 0; e < E; e++) at_off<T>(of + F::out_m(e) * GS, y_off<T, N>(gq, kxi)) = v[e];
    }
    if constexpr (MODE == 0) {
        sfor<0, 3>([&](auto cc) {
            constexpr int c = cc;
            int gq = grp, t0 = 0;
            asm volatile("" : "+v"(gq), "+s"(t0));
            F::template run<NBUF, c != 2>(wr[c], lds, tw + t0, gq, b, cur);
            C2<T>* of = o + size_t(3 + c) * PS;
#pragma unroll
            for (int e = 0; e < E; e++) at_off<T>(of + F::out_m(e) * GS, y_off<T, N>(gq, kxi)) = wr[c][e];
        });
    }
}

// Biot-Savart and the inverse y pass from the vorticity w; `full`: w may hold
// modes outside the sphere, which the vorticity copies then keep.
template <typename T, int N, int MODE, int E_ = Cfg<T, N>::E_BS, int B_ = Cfg<T, N>::B_BS>
__global__ void __launch_bounds__(((N / E_) * B_))
k_bs_inv_y(const C2<T>* __restrict__ w, C2<T>* __restrict__ out, const C2<T>* __restrict__ tw,
           const int* __restrict__ zl, int full, Geom g, size_t bstride) {
    using CF = Cfg<T, N>;
    // box blockIdx.z of a batch of equal boxes bstride elements apart
    w += blockIdx.z * bstride;
    out += blockIdx.z * bstride;
    constexpr int B = B_, E = E_, NT = (N / E_) * B_, NXH = CF::NXH;
    constexpr size_t PS = plane_size(N), GS = (NT / B) * row_stride(N);
    using F = RegFft<T, N, B, B, NT, +1>;
    constexpr int NBUF = fused_bufs<T, N>(B);
    __shared__ C2<T> lds[NBUF * N * B];
    const int tid = threadIdx.x;
    const int b = tid % B, grp = tid / B;
    int tile, kz;
    xcd_tile(tile, kz);
    if (min(kz, N - kz) > zl[tile * B]) return;  // uniform: the whole tile lies outside the sphere
    const int kxi = tile * B + b;
    const double kx = kxi * g.dkx, kzv = kwave(kz, N, g.dkz);
    w += size_t(kz) * NXH;
    C2<T> wr[3][E];
#pragma unroll
    for (int e = 0; e < E; e++) {
        const int n = F::in_row(grp, e);
        const double kyv = kwave(n, N, g.dky);
        const bool in = full || kx * kx + kyv * kyv + kzv * kzv <= g.kM2;
#pragma unroll
        for (int c = 0; c < 3; c++) wr[c][e] = in ? at_off<T>(w + c * PS + F::in_m(e) * GS, y_off<T, N>(grp, kxi)) : mk<T>(T(0), T(0));
    }
    bs_inverse_y<T, N, MODE, F, E, NBUF>(wr, lds, 0, tw, out, grp, b, kxi, kz, g);
}

// ------------------------------------------------------------ generic strided pass (in place)
// element (n, b) of tile (blockIdx.x, blockIdx.y) of plane p of box q
// (blockIdx.z = q * planes + p) at
//   base + q * bstride + p * plane_size(N) + blockIdx.y * ostride + n * estride + kx0 + b
// Tile shape: B columns, E complex values per thread (N / E threads per
// column); the shapes a context may use are listed by pass_shapes() and
// picked by the pass autotuner.
// BAND: the z pass of the step, which moves the rows within the band table zl
// only: the inverse pass takes the rows beyond as zero, the forward pass does
// not store them, and columns with no row in the band are left alone.
template <int N> BFPSH_DEV bool in_band(int n, int lim) { return min(n, N - n) <= lim; }

template <typename T, int N, int SIGN, int E, int B, bool BAND>
__global__ void __launch_bounds__((N / E) * B)
k_pass(C2<T>* __restrict__ data, size_t estride, size_t ostride, const C2<T>* __restrict__ tw, int planes,
       size_t bstride, const int* __restrict__ zl) {
    constexpr int NT = (N / E) * B;
    using F = RegFft<T, N, B, B, NT, SIGN>;
    static_assert(F::E == E, "tile shape");
    constexpr size_t PS = plane_size(N);
    __shared__ C2<T> lds[N * B];
    const int tid = threadIdx.x;
    const int b = tid % B, grp = tid / B;
    int lim = N;
    if constexpr (BAND) {
        if (zl[blockIdx.x * B] < 0) return;  // uniform
        lim = zl[blockIdx.x * B + b];
    }
    // blockIdx.z = box * planes + plane (boxes bstride elements apart)
    const int box = blockIdx.z / planes, plane = blockIdx.z % planes;
    C2<T>* base = data + box * bstride + plane * PS + blockIdx.y * ostride + blockIdx.x * B;
    const uint32_t off = (uint32_t(grp) * uint32_t(estride) + uint32_t(b)) * uint32_t(sizeof(C2<T>));
    const size_t gs = F::G * estride;
    C2<T> v[E];
#pragma unroll
    for (int e = 0; e < E; e++) {
        const int n = F::in_row(grp, e);
        const C2<T>* row = base + F::in_m(e) * gs;
        if constexpr (BAND && SIGN > 0) v[e] = in_band<N>(n, lim) ? at_off<T>(row, off) : mk<T>(T(0), T(0));
        else v[e] = at_off<T>(row, off);
    }
    int cur = 0;
    F::template run<1, false>(v, lds, tw, grp, b, cur);
    if constexpr (BAND && SIGN < 0) {
        // (not to be sunk into the conditional stores)
#pragma unroll
        for (int e = 0; e < E; e++) asm volatile("" : "+v"(v[e].x), "+v"(v[e].y));
    }
#pragma unroll
    for (int e = 0; e < E; e++) {
        const int n = F::out_row(grp, e);
        if (!(BAND && SIGN < 0) || in_band<N>(n, lim)) at_off<T>(base + F::out_m(e) * gs, off) = v[e];
    }
}

// Persistent form of k_pass: gridDim.x workgroups (as many as fit on the
// chip at once) each walk tiles t = blockIdx.x + k gridDim.x of the
// ntx x nty x (planes x boxes) tile grid, and load the columns of their
// next tile while the current one is transformed and stored, so that
// global-memory latency hides behind the FFT (the barriers of the FFT
// order LDS only and leave those loads in flight).
template <typename T, int N, int SIGN, int E, int B, bool BAND>
__global__ void __launch_bounds__((N / E) * B)
k_pass_pp(C2<T>* __restrict__ data, size_t estride, size_t ostride, const C2<T>* __restrict__ tw, int planes,
          size_t bstride, const int* __restrict__ zl, int ntx, int nty, int ntiles) {
    constexpr int NT = (N / E) * B;
    using F = RegFft<T, N, B, B, NT, SIGN>;
    static_assert(F::E == E, "tile shape");
    constexpr size_t PS = plane_size(N);
    __shared__ C2<T> lds[N * B];
    const int tid = threadIdx.x;
    const int b = tid % B, grp = tid / B;
    // tile t: its column's address and (BAND) band limit
    auto base_of = [&](int t, int& lim) {
        const int x = t % ntx, r = t / ntx, y = r % nty, zp = r / nty;
        const int box = zp / planes, plane = zp % planes;
        lim = BAND ? zl[x * B + b] : N;
        return data + box * bstride + plane * PS + size_t(y) * ostride + size_t(x) * B;
    };
    const uint32_t off = (uint32_t(grp) * uint32_t(estride) + uint32_t(b)) * uint32_t(sizeof(C2<T>));
    const size_t gs = F::G * estride;
    auto load = [&](const C2<T>* p, int lim, C2<T> (&v)[E]) {
#pragma unroll
        for (int e = 0; e < E; e++) {
            const int n = F::in_row(grp, e);
            const C2<T>* row = p + F::in_m(e) * gs;
            if constexpr (BAND && SIGN > 0) v[e] = in_band<N>(n, lim) ? at_off<T>(row, off) : mk<T>(T(0), T(0));
            else v[e] = at_off<T>(row, off);
        }
    };
    int t = blockIdx.x;
    if (t >= ntiles) return;
    int lim, nlim = 0;
    C2<T>* p = base_of(t, lim);
    C2<T>* pn = nullptr;
    C2<T> cur[E], nxt[E];
    load(p, lim, cur);
    for (;;) {
        const int tn = t + int(gridDim.x);
        const bool more = tn < ntiles;  // uniform
        if (more) {
            pn = base_of(tn, nlim);
            load(pn, nlim, nxt);
        }
        int buf = 0;
        F::template run<1, true>(cur, lds, tw, grp, b, buf);
#pragma unroll
        for (int e = 0; e < E; e++) {
            const int n = F::out_row(grp, e);
            if (!BAND || (SIGN > 0 ? lim >= 0 : in_band<N>(n, lim))) at_off<T>(p + F::out_m(e) * gs, off) = cur[e];
        }
        if (!more) break;
#pragma unroll
        for (int e = 0; e < E; e++) cur[e] = nxt[e];
        t = tn;
        p = pn;
        lim = nlim;
    }
}

// Tile shapes (E values per thread, B columns, pp: the persistent
// prefetching form) of the plain strided pass for one (precision, N): the
// built-in choice (Cfg) first, then, for N >= 256 (below that a box is
// cache-resident and launch-bound), every shape with E in {8, 12, 16, 24,
// 32} dividing N with a radix plan, B dividing N/2, 64..1024 threads, at
// least 32-byte row segments and at most 128 KB of LDS, and the persistent
// form of each whose two register tiles (4 E registers of FP32, 8 E of
// FP64) take at most 2/5 of a lane's registers (beyond that it spills) --
// up to kMaxPassShapes in all.
struct PassShape {
    int e, b, pp;
};
constexpr int kMaxPassShapes = 16;
struct PassShapes {
    int n;
    PassShape v[kMaxPassShapes];
};
template <typename T, int N>
constexpr PassShapes pass_shapes() {
    using CF = Cfg<T, N>;
    PassShapes s{};
    s.n = 0;
    s.v[s.n++] = PassShape{CF::E_PASS, CF::B, 0};
    if (N < 256) return s;
    constexpr int es[5] = {8, 12, 16, 24, 32};
    constexpr int bs[6] = {2, 4, 8, 16, 32, 64};
    for (int pp = 0; pp < 2; pp++)
        for (int i = 0; i < 5; i++) {
            const int e = es[i];
            if (N % e != 0 || make_plan_e(N, e).ns <= 0) continue;
            for (int j = 0; j < 6; j++) {
                const int b = bs[j];
                const long nt = long(N / e) * b;
                if ((N / 2) % b != 0 || nt < 64 || nt > 1024) continue;
                // persistent form: its two register tiles at most 2/5 of the
                // registers a lane gets (256, or 128 in 1024-thread workgroups)
                if (pp && 5 * (2 * e * int(sizeof(C2<T>)) / 4) > 2 * (nt > 512 ? 128 : 256)) continue;
                if (long(N) * b * long(sizeof(C2<T>)) > 131072 || b * int(sizeof(C2<T>)) < 32) continue;
                bool dup = false;
                for (int k = 0; k < s.n; k++) dup |= s.v[k].e == e && s.v[k].b == b && s.v[k].pp == pp;
                if (dup || s.n == kMaxPassShapes) continue;
                s.v[s.n++] = PassShape{e, b, pp};
            }
        }
    return s;
}

// Tile shapes of the fused first (Biot-Savart + inverse y) and last
// (forward y + update) passes, which hold three components in registers:
// the built-in choice first, then for N >= 512 the shapes with E in
// {8, 16}, 64..1024 threads, at least 64-byte row segments, at most 128 KB
// of LDS, and three components of E values that take at most 96 registers
// of a lane (48 in 1024-thread workgroups, whose lanes get 128 registers):
// larger shapes spill.
template <typename T, int N>
constexpr PassShapes fused_shapes(int e0, int b0) {
    PassShapes s{};
    s.n = 0;
    s.v[s.n++] = PassShape{e0, b0, 0};
    if (N < 512) return s;
    constexpr int es[2] = {8, 16};
    constexpr int bs[4] = {4, 8, 16, 32};
    for (int i = 0; i < 2; i++)
        for (int j = 0; j < 4; j++) {
            const int e = es[i], b = bs[j];
            const long nt = long(N / e) * b;
            if (N % e != 0 || (N / 2) % b != 0 || nt < 64 || nt > 1024) continue;
            if (long(N) * b * long(sizeof(C2<T>)) > 131072 || b * int(sizeof(C2<T>)) < 64) continue;
            const int regs = 3 * e * int(sizeof(C2<T>)) / 4;  // VGPRs of the three components
            if (regs > (nt > 512 ? 48 : 96)) continue;  // beyond these the compiler spills
            bool dup = false;
            for (int k = 0; k < s.n; k++) dup |= s.v[k].e == e && s.v[k].b == b;
            if (dup || s.n == kMaxPassShapes) continue;
            s.v[s.n++] = PassShape{e, b, 0};
        }
    return s;
}

// ------------------------------------------------------------ x passes on row pairs
// Row pair q of row block: rows (y, z = 2q) and (y, z = 2q+1) of a plane.
// Inverse: Z[k] = A[k] + i B[k] (k < N/2; k = 0 real parts only, as a c2r
// ignores the imaginary part of the zero mode), Z[N/2] = 0,
// Z[N-k] = conj(A[k]) + i conj(B[k]); z = IDFT(Z); row z = Re z, row z+1 = Im z.
// Forward: Z = DFT(a + i b); A[k] = (Z[k] + conj Z[N-k]) / 2,
// B[k] = (Z[k] - conj Z[N-k]) / (2 i).
// NCOL columns at once: all global loads of a thread are issued before its
// LDS stores.  Column col reads rows ra(col), rb(col) = base + off[col].
// Modes k > xl lie outside the dealiasing sphere: taken as zero, not read.
template <typename T, int N, int LS, int NCOL, int NT>
BFPSH_DEV void rows_unpack_inverse(C2<T>* lds, const C2<T>* const (&ra)[NCOL], const C2<T>* const (&rb)[NCOL],
                                   int xl, int tid) {
    constexpr int H = N / 2;
    constexpr int PER = (H + NT - 1) / NT;
#pragma unroll
    for (int it = 0; it < PER; it++) {
        const int k = tid + it * NT;
        if (H % NT != 0 && k >= H) break;
        C2<T> A[NCOL], Bv[NCOL];
#pragma unroll
        for (int col = 0; col < NCOL; col++) {
            A[col] = k <= xl ? ra[col][k] : mk<T>(T(0), T(0));
            Bv[col] = k <= xl ? rb[col][k] : mk<T>(T(0), T(0));
        }
#pragma unroll
        for (int col = 0; col < NCOL; col++) {
            if (k == 0) {
                lds[col] = mk<T>(A[col].x, Bv[col].x);
                lds[H * LS + col] = mk<T>(T(0), T(0));
            } else {
                lds[k * LS + col] = mk<T>(A[col].x - Bv[col].y, A[col].y + Bv[col].x);
                lds[(N - k) * LS + col] = mk<T>(A[col].x + Bv[col].y, Bv[col].x - A[col].y);
            }
        }
    }
}
template <typename T, int N, int LS>
BFPSH_DEV void rows_pack_forward(const C2<T>* lds, int col, C2<T>* ra, C2<T>* rb, int xl, int tid, int nt) {
    constexpr int H = N / 2;
    for (int k = tid; k < min(H, xl + 1); k += nt) {
        const C2<T> Z = lds[k * LS + col];
        const C2<T> M = lds[((N - k) % N) * LS + col];
        ra[k] = mk<T>(T(0.5) * (Z.x + M.x), T(0.5) * (Z.y - M.y));
        rb[k] = mk<T>(T(0.5) * (Z.y + M.y), T(-0.5) * (Z.x - M.x));
    }
}

// u x omega / N^3 in real space between the inverse and forward x passes
// (omega_nonlin, bfps/cpp/vorticity_equation.cpp:297-323).
// in:  planes 0..2 = u_hat, 3..5 = omega_hat after the z and y inverse passes
// out: planes 0..2 = x-transformed (u x omega)/N^3 (in place); optional real
//      velocity ru (3 real planes [y][z][x]) for the tracers.
template <typename T, int N>
__global__ void __launch_bounds__((Cfg<T, N>::NT_ROW))
k_rows_cross(C2<T>* __restrict__ data, T* __restrict__ ru, const C2<T>* __restrict__ tw, const int* __restrict__ zl,
             T npoints, size_t bstride) {
    using CF = Cfg<T, N>;
    // LDS row stride: odd, so lanes striding by rows hit distinct banks
    constexpr int RP = CF::RP, NT = CF::NT_ROW, NXH = CF::NXH, LS = CF::LS_ROW;
    constexpr size_t PS = plane_size(N), YS = row_stride(N);
    __shared__ C2<T> lds[N * LS];
    // box blockIdx.y of a batch (complex planes and real velocity move together)
    data += blockIdx.y * bstride;
    if (ru) ru += blockIdx.y * 2 * bstride;
    // the 1/npoints normalization as a product (exact for the power-of-two
    // sizes, within an ulp of the quotient otherwise)
    const T inp = T(1) / npoints;
    const int xl = zl[NXH];
    const int tid = threadIdx.x;
    const int q0 = blockIdx.x * RP;  // first row pair; rows (y, z) flattened: row = y*N + z
    {
        const C2<T>* ra[6 * RP];
        const C2<T>* rb[6 * RP];
#pragma unroll
        for (int c = 0; c < 6; c++)
#pragma unroll
            for (int p = 0; p < RP; p++) {
                const size_t row = size_t(q0 + p) * 2;
                ra[c * RP + p] = data + c * PS + crow<N>(row);
                rb[c * RP + p] = data + c * PS + crow<N>(row) + NXH;
            }
        rows_unpack_inverse<T, N, LS, 6 * RP, NT>(lds, ra, rb, xl, tid);
    }
    __syncthreads();
    fft_tile<T, N, 6 * RP, LS, NT, CF::RMAX, +1>(lds, tw, tid);
    for (int e = tid; e < N * RP; e += NT) {
        const int nn = e / RP, p = e % RP;
        C2<T> u[3], w[3];
#pragma unroll
        for (int c = 0; c < 3; c++) {
            u[c] = lds[nn * LS + c * RP + p];
            w[c] = lds[nn * LS + (3 + c) * RP + p];
        }
        if (ru) {
            const size_t row = size_t(q0 + p) * 2;
#pragma unroll
            for (int c = 0; c < 3; c++) {
                ru[c * 2 * PS + rrow<N>(row) + nn] = u[c].x;
                ru[c * 2 * PS + rrow<N>(row) + N + nn] = u[c].y;
            }
        }
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const int c1 = (c + 1) % 3, c2 = (c + 2) % 3;
            const T re = u[c1].x * w[c2].x - u[c2].x * w[c1].x;
            const T im = u[c1].y * w[c2].y - u[c2].y * w[c1].y;
            lds[nn * LS + c * RP + p] = mk<T>(re * inp, im * inp);
        }
    }
    __syncthreads();
    fft_tile<T, N, 3 * RP, LS, NT, CF::RMAX, -1>(lds, tw, tid);
    for (int c = 0; c < 3; c++)
        for (int p = 0; p < RP; p++) {
            const size_t row = size_t(q0 + p) * 2;
            rows_pack_forward<T, N, LS>(lds, c * RP + p, data + c * PS + crow<N>(row),
                                        data + c * PS + crow<N>(row) + NXH, xl, tid, NT);
        }
}

// Register-resident form of k_rows_cross (FP32, N <= 512): G = N / 8 threads
// own one row pair and hold 8 values of each of the six components, so the
// cross product is formed in registers; the radix exchanges of each
// component go through an LDS region private to the row pair (with padding
// slots against bank conflicts), and the pairing of Z[k] with Z[N-k] in the packed
// rows is a lane shuffle.  A row pair lives inside one wave (G <= 64), so the
// exchanges need wave-level ordering only, no workgroup barrier.  Element e
// of a thread holds row g + G sigma(e) at the input of the FFT and row
// g + G tau(e) at its output (g = thread index within the row pair).
template <typename T, int N>
struct RowsW {
    static constexpr int E = 8, G = N / E, NT = 256, RPB = NT / G, H = E / 2;
    static constexpr int PAD = BFPSH_RW_PAD;  // one LDS slot of padding every 2^PAD rows
    static constexpr int SL = N + (N >> PAD);  // LDS slots per row pair
    static constexpr bool ok = sizeof(T) == 4 && N >= 64 && N <= 512 && (N & (N - 1)) == 0;
    using P = PlanE<N, E>;
    static constexpr int S = P::nstages;
    static constexpr int sigma(int e) {
        const int R = P::radix(0);
        return e / R + (e % R) * (E / R);
    }
    static constexpr int tau(int e) {
        const int R = P::radix(S - 1);
        return e / R + (e % R) * (E / R);
    }
    static constexpr int tau_inv(int m) {
        for (int e = 0; e < E; e++)
            if (tau(e) == m) return e;
        return -1;
    }
    static BFPSH_DEV int slot(int row) { return row + (row >> PAD); }
};

BFPSH_DEV void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// FFT of NCG components of a row pair at once (their exchanges share the
// wave-level ordering points): stage inputs in v, outputs in v
template <typename T, int N, int SIGN, int NCG>
BFPSH_DEV void rows_w_fft(C2<T> (&v)[NCG][8], C2<T>* reg, const C2<T>* __restrict__ tw, int g) {
    using RW = RowsW<T, N>;
    using F = RegFft<T, N, 1, 1, RW::G, SIGN>;
    // an opaque twiddle offset: the twiddles are re-read (from cache) per
    // group instead of being held in registers across all of them (an opaque
    // pointer would lose its address space and be read by flat loads)
    int t0 = 0;
    asm volatile("" : "+s"(t0));
    const C2<T>* twl = tw + t0;
    // likewise the LDS slot addresses are recomputed per group
    int gl = g;
    asm volatile("" : "+v"(gl));
    sfor<0, RW::S>([&](auto s) {
#pragma unroll
        for (int c = 0; c < NCG; c++) F::template compute_stage<s>(v[c], twl, gl);
        if constexpr (s + 1 < RW::S) {
#pragma unroll
            for (int c = 0; c < NCG; c++)
#pragma unroll
                for (int e = 0; e < 8; e++) reg[c * RW::SL + RW::slot(F::out_row_s(s, gl, e))] = v[c][e];
            wave_sync();
#pragma unroll
            for (int c = 0; c < NCG; c++)
#pragma unroll
                for (int e = 0; e < 8; e++) v[c][e] = reg[c * RW::SL + RW::slot(F::in_row_s(s + 1, gl, e))];
            wave_sync();
        }
    });
}

template <typename T>
BFPSH_DEV C2<T> shfl2(C2<T> a, int src) {
    return mk<T>(__shfl(a.x, src, 64), __shfl(a.y, src, 64));
}

template <typename T, int N>
__global__ void __launch_bounds__(256, BFPSH_RW_WAVES)
k_rows_cross_w(C2<T>* __restrict__ data, T* __restrict__ ru, const C2<T>* __restrict__ tw,
               const int* __restrict__ zl, T npoints, size_t bstride) {
    using RW = RowsW<T, N>;
    constexpr int E = RW::E, G = RW::G, H = RW::H, RPB = RW::RPB, NXH = N / 2;
    constexpr size_t PS = plane_size(N), YS = row_stride(N);
    static_assert(RW::ok && 64 % G == 0, "row pair inside one wave");
    __shared__ C2<T> lds[RPB * 3 * RW::SL];
    data += blockIdx.y * bstride;
    if (ru) ru += blockIdx.y * 2 * bstride;
    const T inp = T(1) / npoints;  // normalization as a product, as k_rows_cross
    const int xl = zl[NXH];  // modes beyond are zero: neither read nor written
    const int tid = threadIdx.x;
    const int rp = tid / G, g = tid % G;
    const int partner = (tid & 63) - g + (G - g) % G;  // lane holding index N - k
    C2<T>* reg = lds + rp * 3 * RW::SL;
    const size_t q = size_t(blockIdx.x) * RPB + rp;  // rows 2q, 2q + 1 (row = y N + z)
    const size_t ra = crow<N>(2 * q), rb = ra + NXH;
    C2<T> v[6][E];
    // unpack (as rows_unpack_inverse): Z[k] = A[k] + i B[k], Z[N/2] = 0,
    // Z[N-k] = conj(A[k]) + i conj(B[k]); rows k = g + G m, m < E / 2.  The
    // loads of omega are issued before the FFTs of u.
    C2<T> A[3][H], B[3][H];
    auto load = [&](int c0) {
#pragma unroll
        for (int c = 0; c < 3; c++)
#pragma unroll
            for (int m = 0; m < H; m++) {
                const bool in = g + G * m <= xl;
                A[c][m] = in ? data[(c0 + c) * PS + ra + g + G * m] : mk<T>(T(0), T(0));
                B[c][m] = in ? data[(c0 + c) * PS + rb + g + G * m] : mk<T>(T(0), T(0));
            }
    };
    auto unpack = [&](C2<T> (&vv)[3][E]) {
#pragma unroll
        for (int c = 0; c < 3; c++) {
            C2<T> z[E];
#pragma unroll
            for (int m = 0; m < H; m++) {
                z[m] = mk<T>(A[c][m].x - B[c][m].y, A[c][m].y + B[c][m].x);
                if (m == 0 && g == 0) z[m] = mk<T>(A[c][m].x, B[c][m].x);
            }
#pragma unroll
            for (int m = H; m < E; m++) {
                C2<T> a = shfl2<T>(A[c][E - 1 - m], partner), b = shfl2<T>(B[c][E - 1 - m], partner);
                if (g == 0) {
                    if (m == H) {
                        a = mk<T>(T(0), T(0));
                        b = a;
                    } else {
                        a = A[c][(E - m) % H];
                        b = B[c][(E - m) % H];
                    }
                }
                z[m] = mk<T>(a.x + b.y, b.x - a.y);
            }
#pragma unroll
            for (int e = 0; e < E; e++) vv[c][e] = z[RW::sigma(e)];
        }
    };
    C2<T> (&vu)[3][E] = *reinterpret_cast<C2<T>(*)[3][E]>(&v[0][0]);
    C2<T> (&vw)[3][E] = *reinterpret_cast<C2<T>(*)[3][E]>(&v[3][0]);
    load(0);
    unpack(vu);
    load(3);
    rows_w_fft<T, N, +1, 3>(vu, reg, tw, g);
    unpack(vw);
    rows_w_fft<T, N, +1, 3>(vw, reg, tw, g);
    if (ru) {
#pragma unroll
        for (int c = 0; c < 3; c++)
#pragma unroll
            for (int e = 0; e < E; e++) {
                const int x = g + G * RW::tau(e);
                ru[c * 2 * PS + rrow<N>(2 * q) + x] = v[c][e].x;
                ru[c * 2 * PS + rrow<N>(2 * q) + N + x] = v[c][e].y;
            }
    }
    // (u x omega) / N^3 on rows g + G tau(e), reordered to the forward FFT's
    // input rows g + G sigma(e)
    C2<T> f[3][E];
#pragma unroll
    for (int e = 0; e < E; e++) {
        const int eo = RW::tau_inv(RW::sigma(e));
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const int c1 = (c + 1) % 3, c2 = (c + 2) % 3;
            const C2<T> u1 = v[c1][eo], u2 = v[c2][eo], w1 = v[3 + c1][eo], w2 = v[3 + c2][eo];
            const T re = u1.x * w2.x - u2.x * w1.x;
            const T im = u1.y * w2.y - u2.y * w1.y;
            f[c][e] = mk<T>(re * inp, im * inp);
        }
    }
    rows_w_fft<T, N, -1, 3>(f, reg, tw, g);
#pragma unroll
    for (int c = 0; c < 3; c++) {
        // pack (as rows_pack_forward): A[k] = (Z[k] + conj Z[N-k]) / 2,
        // B[k] = (Z[k] - conj Z[N-k]) / (2 i), k = g + G m, m < E / 2
#pragma unroll
        for (int m = 0; m < H; m++) {
            const C2<T> Z = f[c][RW::tau_inv(m)];
            C2<T> M = shfl2<T>(f[c][RW::tau_inv(E - 1 - m)], partner);
            if (g == 0) M = f[c][RW::tau_inv((E - m) % E)];
            if (g + G * m > xl) continue;
            data[c * PS + ra + g + G * m] = mk<T>(T(0.5) * (Z.x + M.x), T(0.5) * (Z.y - M.y));
            data[c * PS + rb + g + G * m] = mk<T>(T(0.5) * (Z.y + M.y), T(-0.5) * (Z.x - M.x));
        }
    }
}

// Small boxes: the middle of a stage in one launch.  A workgroup holds the
// (z, x) slab of one y: inverse z pass, c2r x pass, cross product, r2c x pass
// and forward z pass of k_pass, k_rows_cross and k_pass above, with the same
// band.  At these sizes each of the three launches takes 3 to 12 us for a
// fraction of a microsecond of traffic: what bounds them is launch and
// latency, once instead of three times here.  A plane of the slab passes
// through LDS; the real values of the six components stay in registers.
// Every pass of data through LDS alternates between two tiles (one barrier
// each).  Threads hold E values; along z, thread (g, b) holds column b with b
// fastest; along x, thread (q, g) holds row pair q with g fastest.
template <typename T, int N>
struct Slab {
    // Whole steps, three launches a stage -> one: 16^3 64 -> 53 us, 32^3 71 ->
    // 69 us, 64^3 FP32 116 -> 105 us.  Not in FP64 at 64^3 (one workgroup a CU
    // for a chain twice as long, 127 -> 135 us) nor at 48^3 (four short radix
    // stages along each axis, 103 -> 111 us FP32, 115 -> 137 us FP64)
    static constexpr bool ok = N <= 32 || (sizeof(T) == 4 && N == 64);
    static constexpr int E = N == 16 ? 2 : 4;
    static constexpr int H = N / 2, G = N / E, NT = G * H;
    static constexpr int XS = N + 1;       // row pairs of a tile along x
    static constexpr int TILE = H * XS;    // complex values (the z layout [N][H] is smaller)
    // components that share the exchanges, as LDS allows
    static constexpr int NC = 3;
    static_assert(!ok || 2 * NC * TILE * int(sizeof(C2<T>)) <= 131072, "two tiles of three components");
};

template <typename T, int N>
__global__ void __launch_bounds__((Slab<T, N>::NT))
k_slab_cross(C2<T>* __restrict__ data, T* __restrict__ ru, const C2<T>* __restrict__ tw, const int* __restrict__ zl,
             T npoints, size_t bstride) {
    using SB = Slab<T, N>;
    constexpr int E = SB::E, H = SB::H, G = SB::G, NT = SB::NT, XS = SB::XS, TILE = SB::TILE;
    constexpr int NC = SB::NC;
    constexpr size_t PS = plane_size(N), YS = row_stride(N);
    using ZI = RegFft<T, N, H, H, NT, +1>;
    using ZF = RegFft<T, N, H, H, NT, -1>;
    using XI = RegFft<T, N, 1, 1, G, +1>;
    using XF = RegFft<T, N, 1, 1, G, -1>;
    static_assert(ZI::E == E && XI::E == E, "values per thread");
    __shared__ C2<T> lds[2][NC][TILE];
    const int y = blockIdx.x, tid = threadIdx.x;
    data += blockIdx.y * bstride + size_t(y) * YS;
    if (ru) ru += blockIdx.y * 2 * bstride + size_t(y) * 2 * YS;
    const T inp = T(1) / npoints;
    const int b = tid % H, gz = tid / H;   // along z
    const int gx = tid % G, q = tid / G;   // along x
    const int lim = zl[b];
    int cur = 0;
    // exchange between stage s and s + 1 of the FFTs of NC components: element
    // addresses by the stage's output and input rows
    auto exchange = [&](C2<T> (&v)[NC][E], auto&& out_at, auto&& in_at) {
#pragma unroll
        for (int c = 0; c < NC; c++)
#pragma unroll
            for (int e = 0; e < E; e++) lds[cur][c][out_at(e)] = v[c][e];
        __syncthreads();
#pragma unroll
        for (int c = 0; c < NC; c++)
#pragma unroll
            for (int e = 0; e < E; e++) v[c][e] = lds[cur][c][in_at(e)];
        cur ^= 1;
    };
    auto fft_z = [&](C2<T> (&v)[NC][E], auto f) {
        using F = decltype(f);
        sfor<0, F::S>([&](auto s) {
#pragma unroll
            for (int c = 0; c < NC; c++) F::template compute_stage<s>(v[c], tw, gz);
            if constexpr (s + 1 < F::S)
                exchange(v, [&](int e) { return F::out_row_s(s, gz, e) * H + b; },
                         [&](int e) { return F::in_row_s(s + 1, gz, e) * H + b; });
        });
    };
    auto fft_x = [&](C2<T> (&v)[NC][E], auto f) {
        using F = decltype(f);
        sfor<0, F::S>([&](auto s) {
#pragma unroll
            for (int c = 0; c < NC; c++) F::template compute_stage<s>(v[c], tw, gx);
            if constexpr (s + 1 < F::S)
                exchange(v, [&](int e) { return q * XS + F::out_row_s(s, gx, e); },
                         [&](int e) { return q * XS + F::in_row_s(s + 1, gx, e); });
        });
    };
    C2<T> val[6][E];
    sfor<0, 6 / NC>([&](auto gi) {
        constexpr int c0 = gi * NC;
        C2<T> v[NC][E];
#pragma unroll
        for (int c = 0; c < NC; c++)
#pragma unroll
            for (int e = 0; e < E; e++) {
                const int n = ZI::in_row(gz, e);
                v[c][e] = in_band<N>(n, lim) ? data[(c0 + c) * PS + size_t(n) * H + b] : mk<T>(T(0), T(0));
            }
        fft_z(v, ZI{});
#pragma unroll
        for (int c = 0; c < NC; c++)
#pragma unroll
            for (int e = 0; e < E; e++) lds[cur][c][ZI::out_row(gz, e) * H + b] = v[c][e];
        __syncthreads();
        // rows 2q and 2q + 1 packed, as rows_unpack_inverse
#pragma unroll
        for (int c = 0; c < NC; c++)
#pragma unroll
            for (int e = 0; e < E; e++) {
                const int k = XI::in_row(gx, e), kk = k < H ? k : N - k;
                const C2<T> A = lds[cur][c][2 * q * H + (k == H ? 0 : kk)];
                const C2<T> Bv = lds[cur][c][(2 * q + 1) * H + (k == H ? 0 : kk)];
                C2<T> z = k < H ? mk<T>(A.x - Bv.y, A.y + Bv.x) : mk<T>(A.x + Bv.y, Bv.x - A.y);
                if (k == 0) z = mk<T>(A.x, Bv.x);
                if (k == H) z = mk<T>(T(0), T(0));
                v[c][e] = z;
            }
        cur ^= 1;
        fft_x(v, XI{});
#pragma unroll
        for (int c = 0; c < NC; c++)
#pragma unroll
            for (int e = 0; e < E; e++) val[c0 + c][e] = v[c][e];
    });
    if (ru) {
#pragma unroll
        for (int c = 0; c < 3; c++)
#pragma unroll
            for (int e = 0; e < E; e++) {
                T* r = ru + c * 2 * PS + 2 * q * N + XI::out_row(gx, e);
                r[0] = val[c][e].x;
                r[N] = val[c][e].y;
            }
    }
    // (u x omega) / N^3 on rows gx + G out_m(e), reordered to the forward
    // FFT's input rows
    C2<T> f[3][E];
    sfor<0, E>([&](auto e) {
        sfor<0, E>([&](auto i) {
            if constexpr (XI::out_m(i) == XF::in_m(e)) {
#pragma unroll
                for (int c = 0; c < 3; c++) {
                    const int c1 = (c + 1) % 3, c2 = (c + 2) % 3;
                    const C2<T> u1 = val[c1][i], u2 = val[c2][i], w1 = val[3 + c1][i], w2 = val[3 + c2][i];
                    f[c][e] = mk<T>((u1.x * w2.x - u2.x * w1.x) * inp, (u1.y * w2.y - u2.y * w1.y) * inp);
                }
            }
        });
    });
    fft_x(f, XF{});
#pragma unroll
    for (int c = 0; c < NC; c++)
#pragma unroll
        for (int e = 0; e < E; e++) lds[cur][c][q * XS + XF::out_row(gx, e)] = f[c][e];
    __syncthreads();
    // the rows' spectra, as rows_pack_forward: even z from A, odd from B
#pragma unroll
    for (int c = 0; c < NC; c++)
#pragma unroll
        for (int e = 0; e < E; e++) {
            const int z = ZF::in_row(gz, e);
            const C2<T>* row = &lds[cur][c][(z / 2) * XS];
            const C2<T> Z = row[b], M = row[(N - b) % N];
            f[c][e] = z % 2 == 0 ? mk<T>(T(0.5) * (Z.x + M.x), T(0.5) * (Z.y - M.y))
                                 : mk<T>(T(0.5) * (Z.y + M.y), T(-0.5) * (Z.x - M.x));
        }
    cur ^= 1;
    fft_z(f, ZF{});
#pragma unroll
    for (int c = 0; c < NC; c++)
#pragma unroll
        for (int e = 0; e < E; e++) {
            const int n = ZF::out_row(gz, e);
            if (in_band<N>(n, lim)) data[c * PS + size_t(n) * H + b] = f[c][e];
        }
}

// c2r x pass of NC planes into real planes out ([y][z][x] each), components
// in groups of up to 3.  out may equal data (in place: a real row occupies
// the bytes of the spectral row with the same index, and a block reads all
// of its rows before writing them).
template <typename T, int N, int NC>
__global__ void __launch_bounds__((Cfg<T, N>::NT_ROW))
k_rows_c2r(const C2<T>* data, T* out, const C2<T>* __restrict__ tw, int xl) {
    using CF = Cfg<T, N>;
    constexpr int NG = NC < 3 ? NC : 3;
    constexpr int RP = CF::RP, NT = CF::NT_ROW, NXH = CF::NXH, LS = NG * RP + 1;
    constexpr size_t PS = plane_size(N), YS = row_stride(N);
    static_assert(NC % NG == 0, "component groups");
    __shared__ C2<T> lds[N * LS];
    const int tid = threadIdx.x;
    const int q0 = blockIdx.x * RP;
    for (int c0 = 0; c0 < NC; c0 += NG) {
        {
            const C2<T>* ra[NG * RP];
            const C2<T>* rb[NG * RP];
#pragma unroll
            for (int c = 0; c < NG; c++)
#pragma unroll
                for (int p = 0; p < RP; p++) {
                    const size_t row = size_t(q0 + p) * 2;
                    ra[c * RP + p] = data + (c0 + c) * PS + crow<N>(row);
                    rb[c * RP + p] = data + (c0 + c) * PS + crow<N>(row) + NXH;
                }
            rows_unpack_inverse<T, N, LS, NG * RP, NT>(lds, ra, rb, xl, tid);
        }
        __syncthreads();
        fft_tile<T, N, NG * RP, LS, NT, CF::RMAX, +1>(lds, tw, tid);
        for (int e = tid; e < N * NG * RP; e += NT) {  // consecutive lanes: consecutive x
            const int col = e / N, nn = e % N;
            const int c = col / RP, p = col % RP;
            const size_t row = size_t(q0 + p) * 2;
            const C2<T> v = lds[nn * LS + col];
            out[(c0 + c) * 2 * PS + rrow<N>(row) + nn] = v.x;
            out[(c0 + c) * 2 * PS + rrow<N>(row) + N + nn] = v.y;
        }
        __syncthreads();
    }
}

// r2c x pass of NC real planes ([y][z][x]) into spectral rows (kx < N/2),
// components in groups of up to 3; out may equal data (in place).
template <typename T, int N, int NC>
__global__ void __launch_bounds__((Cfg<T, N>::NT_ROW))
k_rows_r2c(const T* data, C2<T>* out, const C2<T>* __restrict__ tw) {
    using CF = Cfg<T, N>;
    constexpr int NG = NC < 3 ? NC : 3;
    constexpr int RP = CF::RP, NT = CF::NT_ROW, NXH = CF::NXH, LS = NG * RP + 1;
    constexpr size_t PS = plane_size(N), YS = row_stride(N);
    static_assert(NC % NG == 0, "component groups");
    __shared__ C2<T> lds[N * LS];
    const int tid = threadIdx.x;
    const int q0 = blockIdx.x * RP;
    for (int c0 = 0; c0 < NC; c0 += NG) {
        for (int e = tid; e < N * NG * RP; e += NT) {  // consecutive lanes: consecutive x
            const int col = e / N, nn = e % N;
            const int c = col / RP, p = col % RP;
            const size_t row = size_t(q0 + p) * 2;
            lds[nn * LS + col] = mk<T>(data[(c0 + c) * 2 * PS + rrow<N>(row) + nn],
                                       data[(c0 + c) * 2 * PS + rrow<N>(row) + N + nn]);
        }
        __syncthreads();
        fft_tile<T, N, NG * RP, LS, NT, CF::RMAX, -1>(lds, tw, tid);
        for (int c = 0; c < NG; c++)
            for (int p = 0; p < RP; p++) {
                const size_t row = size_t(q0 + p) * 2;
                rows_pack_forward<T, N, LS>(lds, c * RP + p, out + (c0 + c) * PS + crow<N>(row),
                                            out + (c0 + c) * PS + crow<N>(row) + NXH, N, tid, NT);
            }
        __syncthreads();
    }
}

// ------------------------------------------------------------ integrating factor
// exp(x + y) from a part a, ra of x and b, rb of y, which depend on fewer
// indexes than their sum.  While the factors stay above exp(-1/2) (`slow`,
// uniform; one = 1), a = exp(x) - 1, ra = 0 and the factor is 1 + (a + b + a b),
// whose error is that of its last rounding, like an exponential's own.  Beyond
// (one = 0), that sum would cancel, and a product of two rounded exponentials
// has 1.3 times an exponential's error: there exp(x) = a (1 + ra), a its rounded
// value and ra the rest, from x = m ln 2 + r, |r| <= ln 2 / 2 (argument
// reduction of Cody and Waite) and exp(r) - 1, and the factor a b + a b (ra +
// rb).  The rest is relative, so that it neither over- nor underflows in 32 bits.
// FP64 decay at 64^3 over 64 steps, mean error of a mode at nu dt kM^2 = 1.4 /
// 3: 7.8e-15 / 1.00e-14; by products 1.02e-14 / 1.29e-14; with one rounded
// exponential a factor 8.3e-15 / 9.7e-15.
BFPSH_DEV double if_part(double x, bool slow, float& rest) {
    double q = 0.0;
    if (!slow) {
        q = rint(fmin(fmax(x * 0x1.71547652b82fep+0, -1e9), 1e9));  // x / ln 2
        // (ln 2 and what its rounding leaves)
        x = fma(-q, 0x1.abc9e3b39803fp-56, fma(-q, 0x1.62e42fefa39efp-1, x));
    }
    const double e = expm1(x);
    rest = 0.0f;
    if (slow) return e;
    const double h = 1.0 + e;
    if (h > 0.0) rest = float((e - (h - 1.0)) / h);
    return ldexp(h, int(q));
}
// `one` plus the absolute rest of a part: 1 if slow
BFPSH_DEV double if_rest(double a, float ra, double one) { return fma(double(ra), a, one); }
BFPSH_DEV double if_of(double a, double la, double b, double lb, double one) {
    return one + fma(a, b, fma(a, lb, la * b));
}

// ------------------------------------------------------------ last forward pass + update
// STAGE 1..3 of the integrating-factor SSP-RK3 step
// (vorticity_equation::step, bfps/cpp/vorticity_equation.cpp:358-439), fused
// with the tail of omega_nonlin (:323-355): dealias (kspace.cpp:461-485),
// curl, forcing (:241-288), force_divfree (kspace.cpp:487-519).
// w: planes 0..2 hold the output of the z forward pass ([y][kz][kx]).
// v0 = omega(t); vp = previous stage (stage 2: v1, stage 3: v2); dst receives
// the new stage (stage 3 writes v0 in place and applies the final projection).
// Stages 1 and 2 go on with the first pass of the next stage while its
// vorticity is in registers: Biot-Savart and the inverse y pass into planes
// 0..5 of w (a workgroup reads its columns before it writes them).  That
// saves reading the new vorticity back (3 N^3) and one launch a stage.
//
// Outside the sphere the stages are zero and stay unwritten (v1 and v2 start
// as zeros); stage 3 keeps v0 there, projected, when `full` says that it may
// hold something.  The integrating factor exp(-nu k^2 dt c) is combined from
// one value per ky, in an LDS table, and one per thread for its (kx, kz),
// instead of one exponential per mode (two in stage 2): see if_of.
template <typename T, int N, int STAGE, bool BATCH, int E_ = Cfg<T, N>::E_Y3, int B_ = Cfg<T, N>::B_Y3>
__global__ void __launch_bounds__(((N / E_) * B_))
k_y_update(C2<T>* w, const C2<T>* v0, const C2<T>* vp, C2<T>* dst, const C2<T>* __restrict__ tw,
           const int* __restrict__ zl, int full, Geom g, StepParams sp0, size_t bstride,
           const StepParams* __restrict__ spb) {
    using CF = Cfg<T, N>;
    // BATCH: box blockIdx.z of a batch, its fields bstride elements apart and
    // its own physics parameters in spb (a separate instantiation keeps the
    // single-box kernel's registers free of the batch bookkeeping)
    if constexpr (BATCH) {
        w += blockIdx.z * bstride;
        v0 += blockIdx.z * bstride;
        vp += blockIdx.z * bstride;
        dst += blockIdx.z * bstride;
    }
    const StepParams sp = BATCH ? spb[blockIdx.z] : sp0;
    constexpr int B = B_, E = E_, NT = (N / E_) * B_, NXH = CF::NXH;
    constexpr size_t PS = plane_size(N), GS = (NT / B) * row_stride(N);
    using F = RegFft<T, N, B, B, NT, -1>;
    constexpr int NBUF = fused_bufs<T, N>(B);
    __shared__ C2<T> lds[NBUF * N * B];
    __shared__ double ify[STAGE == 2 ? 2 : 1][N];
    __shared__ float ifr[STAGE == 2 ? 2 : 1][N];
    const int tid = threadIdx.x;
    const int b = tid % B, grp = tid / B;
    // tiles narrower than a 128-byte line (1024^3): neighbouring tiles, the
    // two halves of each line, run on the same XCD and share its L2
    int tile = blockIdx.x, kz = blockIdx.y;
    if constexpr (B * sizeof(C2<T>) < 128) xcd_tile(tile, kz);
    const int kza = min(kz, N - kz);
    if (kza > zl[tile * B]) return;  // uniform: the whole tile lies outside the sphere
    const int kxi = tile * B + b;
    const bool col_in = kza <= zl[kxi];
    const size_t kzs = size_t(kz) * NXH;
    v0 += kzs;
    vp += kzs;
    dst += kzs;
    C2<T> res[3][E];
#pragma unroll
    for (int c = 0; c < 3; c++)
#pragma unroll
        for (int e = 0; e < E; e++)
            res[c][e] = col_in ? at_off<T>(w + c * PS + kzs + F::in_m(e) * GS, y_off<T, N>(grp, kxi)) : mk<T>(T(0), T(0));
    const double kx = kxi * g.dkx, kzv = kwave(kz, N, g.dkz);
    const double dt = sp.dt, nud = sp.nu * dt * (STAGE == 1 ? 1.0 : 0.5);
    const bool slow = fabs(nud) * g.kM2 < 0.5;  // uniform
    for (int i = tid; i < N; i += NT) {
        const double k = kwave(i, N, g.dky);
        ify[0][i] = if_part(-nud * k * k, slow, ifr[0][i]);
        if constexpr (STAGE == 2) ify[1][i] = if_part(nud * k * k, slow, ifr[1][i]);
    }
    const double one = slow ? 1.0 : 0.0;
    float rxz, rxz1 = 0.f;
    const double ifxz = if_part(-nud * (kx * kx + kzv * kzv), slow, rxz);
    const double ifxz1 = STAGE == 2 ? if_part(nud * (kx * kx + kzv * kzv), slow, rxz1) : 0.0;
    const double lxz = if_rest(ifxz, rxz, one), lxz1 = if_rest(ifxz1, rxz1, one);
    __syncthreads();
    // one component after the other; an opaque group index and table offset
    // per component, so that twiddles and LDS addresses are not held across,
    // and opaque results, so that the last butterflies are not sunk into the
    // conditional code below (which would keep all their inputs alive)
    int cur = 0;
#pragma unroll
    for (int c = 0; c < 3; c++) {
        int gq = grp, t0 = 0;
        asm volatile("" : "+v"(gq), "+s"(t0));
        F::template run<NBUF, true>(res[c], lds, tw + t0, gq, b, cur);
#pragma unroll
        for (int e = 0; e < E; e++) asm volatile("" : "+v"(res[c][e].x), "+v"(res[c][e].y));
    }
    const double ikM2 = 1.0 / g.kM2;
    const double fk1sq = sp.fk1 * sp.fk1 * (1 + 1e-12);
    // v0 and vp of element i + 1 are requested before element i is computed
    // (few waves fit beside the three components, so their loads must not
    // wait for one another); nothing else of an element is kept across
    C2<T> p0[2][3], p1[2][3];
    auto fetch = [&](int i, C2<T> (&q0)[3], C2<T> (&q1)[3]) {
        int gq = grp;
        asm volatile("" : "+v"(gq));
        const int ky = F::out_row(gq, i);
        const double kyv = kwave(ky, N, g.dky);
        if (kx * kx + kyv * kyv + kzv * kzv <= g.kM2 || (STAGE == 3 && full)) {
            const uint32_t off = y_off<T, N>(gq, kxi);
            const size_t row = F::out_m(i) * GS;
#pragma unroll
            for (int c = 0; c < 3; c++) {
                q0[c] = at_off<T>(v0 + c * PS + row, off);
                if (STAGE > 1) q1[c] = at_off<T>(vp + c * PS + row, off);
            }
        }
    };
    fetch(0, p0[0], p1[0]);
    sfor<0, E>([&](auto ii) {
        constexpr int i = ii;
        if constexpr (i + 1 < E) fetch(i + 1, p0[(i + 1) % 2], p1[(i + 1) % 2]);
        const C2<T>(&w0)[3] = p0[i % 2];
        const C2<T>(&w1)[3] = p1[i % 2];
        int gq = grp;
        asm volatile("" : "+v"(gq));
        const int ky = F::out_row(gq, i);
        const double kyv = kwave(ky, N, g.dky);
        const double k2 = kx * kx + kyv * kyv + kzv * kzv;
        const uint32_t off = y_off<T, N>(gq, kxi);
        C2<T> nv[3];
        bool write = true;
        if (k2 <= g.kM2) {
            // dealias
            C2<T> a[3];
            if (g.smooth) {
                const double r = k2 * ikM2;
                const double r2 = r * r, r4 = r2 * r2, r8 = r4 * r4, r16 = r8 * r8;
                const double flt = exp(-36.0 * (r16 * r2));
#pragma unroll
                for (int c = 0; c < 3; c++) a[c] = mk<T>(T(res[c][i].x * flt), T(res[c][i].y * flt));
            } else {
#pragma unroll
                for (int c = 0; c < 3; c++) a[c] = k2 >= g.kM2 ? mk<T>(T(0), T(0)) : res[c][i];
            }
            // curl: i k x a
            C2<T> cu[3];
            cu[0] = mk<T>(T(-(kyv * a[2].y - kzv * a[1].y)), T(kyv * a[2].x - kzv * a[1].x));
            cu[1] = mk<T>(T(-(kzv * a[0].y - kx * a[2].y)), T(kzv * a[0].x - kx * a[2].x));
            cu[2] = mk<T>(T(-(kx * a[1].y - kyv * a[0].y)), T(kx * a[1].x - kyv * a[0].x));
            // forcing with the stage's source vorticity
            // (the wavenumber's root is taken near the band only)
            if ((sp.forcing == 1 || sp.forcing == 3) && k2 <= fk1sq) {
                const double kn = sqrt(k2);
                if (sp.fk0 <= kn && sp.fk1 >= kn) {
                    const double amp = sp.forcing == 1 ? sp.famp : sp.famp_dev[STAGE - 1];
#pragma unroll
                    for (int c = 0; c < 3; c++) {
                        const C2<T> s = STAGE == 1 ? w0[c] : w1[c];
                        cu[c] = mk<T>(T(cu[c].x + amp * double(s.x) * 1.0), T(cu[c].y + amp * double(s.y) * 1.0));
                    }
                }
            } else if (sp.forcing == 2) {
                if (kxi == 0 && kz == 0 && (ky == sp.fmode || ky == N - sp.fmode))
                    cu[2].x = T(cu[2].x - sp.famp * 1.0 / 2);
            }
            // force_divfree (zero at k = 0), then the integrating-factor RK stage
            const double ik2 = k2 > 0 ? 1.0 / k2 : 0.0;  // one division, then products
            if (k2 > 0) divfree<T>(cu, kx, kyv, kzv, ik2);
            else cu[0] = cu[1] = cu[2] = mk<T>(T(0), T(0));
            const double f0 = if_of(ifxz, lxz, ify[0][ky], if_rest(ify[0][ky], ifr[0][ky], one), one);
#pragma unroll
            for (int c = 0; c < 3; c++) {
                if constexpr (STAGE == 1) {
                    nv[c] = mk<T>(T((w0[c].x + dt * cu[c].x) * f0), T((w0[c].y + dt * cu[c].y) * f0));
                } else if constexpr (STAGE == 2) {
                    const double b1 = ify[STAGE - 1][ky];
                    const double f1 = if_of(ifxz1, lxz1, b1, if_rest(b1, ifr[STAGE - 1][ky], one), one);
                    nv[c] = mk<T>(T((3 * w0[c].x * f0 + (w1[c].x + dt * cu[c].x) * f1) * 0.25),
                                  T((3 * w0[c].y * f0 + (w1[c].y + dt * cu[c].y) * f1) * 0.25));
                } else {
                    const double f3 = f0 * (1.0 / 3);  // products instead of six divisions by 3
                    nv[c] = mk<T>(T((w0[c].x * f0 + 2 * (w1[c].x + dt * cu[c].x)) * f3),
                                  T((w0[c].y * f0 + 2 * (w1[c].y + dt * cu[c].y)) * f3));
                }
            }
            if constexpr (STAGE == 3) {
                // final force_divfree of the new vorticity
                if (k2 > 0) divfree<T>(nv, kx, kyv, kzv, ik2);
                else nv[0] = nv[1] = nv[2] = mk<T>(T(0), T(0));
            }
        } else if (STAGE == 3 && full) {
            // v0 there is kept, with the final projection (k2 > 0)
#pragma unroll
            for (int c = 0; c < 3; c++) nv[c] = w0[c];
            divfree<T>(nv, kx, kyv, kzv, 1.0 / k2);
        } else {
            nv[0] = nv[1] = nv[2] = mk<T>(T(0), T(0));
            write = false;
        }
        if (write) {
#pragma unroll
            for (int c = 0; c < 3; c++) at_off<T>(dst + c * PS + F::out_m(i) * GS, off) = nv[c];
        }
        if constexpr (STAGE < 3) {
#pragma unroll
            for (int c = 0; c < 3; c++) res[c][i] = nv[c];
        }
        __builtin_amdgcn_sched_barrier(0);
    });
    if constexpr (STAGE < 3) {
        // the first inverse pass of the next stage: register element e of
        // its input is row F::in_row(e), which element i of the forward
        // output holds (both are rows grp + G m)
        using FI = RegFft<T, N, B, B, NT, +1>;
        C2<T> wr[3][E];
        sfor<0, E>([&](auto e) {
            sfor<0, E>([&](auto i) {
                if constexpr (F::out_m(i) == FI::in_m(e)) {
#pragma unroll
                    for (int c = 0; c < 3; c++) wr[c][e] = res[c][i];
                }
            });
        });
        bs_inverse_y<T, N, 0, FI, E, NBUF>(wr, lds, cur, tw, w, grp, b, kxi, kz, g);
    }
}

// Fixed energy-injection-rate forcing (not a reference forcing type): the
// linear band forcing with amplitude eps / (2 E_band), E_band = 1/2 sum over
// fk0 <= |k| <= fk1 of nxmodes |omega_hat|^2 / k^2 (= 1/2 sum nxmodes |u_hat|^2
// for solenoidal omega), so that the band gains energy at the rate eps.  One
// block scans the box |k_i| <= fk1 and writes the amplitude to *amp.
template <typename T, int N>
__global__ void __launch_bounds__(256) k_band_amplitude(const C2<T>* __restrict__ w, double* amp, Geom g, double eps,
                                                        double fk0, double fk1, size_t bstride,
                                                        const StepParams* __restrict__ spb, int stage) {
    // box blockIdx.x of a batch: its source field, its own rate, band and
    // amplitude slot (spb[box].famp_dev + stage - 1)
    if (spb) {
        const StepParams& p = spb[blockIdx.x];
        if (p.forcing != 3) return;
        w += blockIdx.x * bstride;
        amp = const_cast<double*>(p.famp_dev) + (stage - 1);
        eps = p.famp;
        fk0 = p.fk0;
        fk1 = p.fk1;
    }
    constexpr int NXH = N / 2;
    constexpr size_t PS = plane_size(N), YS = row_stride(N);
    __shared__ double part[256];
    const int KX = min(NXH - 1, int(fk1 / g.dkx));
    const int KY = min(N / 2 - 1, int(fk1 / g.dky)), KZ = min(N / 2 - 1, int(fk1 / g.dkz));
    const int nyv = 2 * KY + 1, nzv = 2 * KZ + 1;
    const int total = (KX + 1) * nyv * nzv;
    double e = 0.0;
    for (int t = threadIdx.x; t < total; t += 256) {
        const int x = t % (KX + 1), zz = (t / (KX + 1)) % nzv - KZ, yy = t / ((KX + 1) * nzv) - KY;
        const double kx = x * g.dkx, ky = yy * g.dky, kz = zz * g.dkz;
        const double k2 = kx * kx + ky * ky + kz * kz;
        const double kn = sqrt(k2);
        if (!(fk0 <= kn && fk1 >= kn && k2 > 0)) continue;
        const size_t off = size_t(yy < 0 ? yy + N : yy) * YS + size_t(zz < 0 ? zz + N : zz) * NXH + x;
        double m = 0.0;
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const C2<T> v = w[c * PS + off];
            m += double(v.x) * double(v.x) + double(v.y) * double(v.y);
        }
        e += (x == 0 ? 1.0 : 2.0) * m / k2;
    }
    part[threadIdx.x] = e;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (int(threadIdx.x) < s) part[threadIdx.x] += part[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const double eb = 0.5 * part[0];
        *amp = eb > 0 ? eps / (2 * eb) : 0.0;
    }
}

// ------------------------------------------------------------ small spectral kernels
// data of the autotuner's trials: `count` complex values in the unit square
// without a pattern
template <typename T> __global__ void __launch_bounds__(256) k_fill_pattern(C2<T>* d, size_t count) {
    auto value = [](size_t i) { return T(int32_t(uint32_t(i) * 2654435761u)) * T(1.0 / 2147483648.0); };
    for (size_t i = size_t(blockIdx.x) * 256 + threadIdx.x; i < count; i += size_t(gridDim.x) * 256)
        d[i] = mk<T>(value(2 * i), value(2 * i + 1));
}

// field::symmetrize on the kx = 0 plane (bfps/cpp/field.cpp:900-978):
// Im(0,0,0) = 0; (0, kz) = conj(0, N-kz) for N/2 < kz < N;
// (ky, kz) = conj(N-ky, (N-kz) mod N) for N/2 < ky < N.
template <typename T>
__global__ void k_symmetrize(C2<T>* v, int n, int nc, size_t bstride) {
    v += blockIdx.y * bstride;  // box blockIdx.y of a batch
    const int nxh = n / 2;
    const size_t ps = plane_size(n), ys = row_stride(n);
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= n * n) return;
    const int ky = idx / n, kz = idx % n;
    for (int c = 0; c < nc; c++) {
        C2<T>* p = v + c * ps;
        if (ky == 0 && kz == 0) {
            p[0].y = T(0);
        } else if ((ky > n / 2) || (ky == 0 && kz > n / 2)) {
            const C2<T> m = p[size_t((n - ky) % n) * ys + size_t((n - kz) % n) * nxh];
            p[size_t(ky) * ys + size_t(kz) * nxh] = cconj<T>(m);
        }
    }
}

// low_pass(kM) (k^2 >= kM^2 -> 0) followed by force_divfree
// (io_checkpoint read projections, bfps/cpp/vorticity_equation.hpp:118-127)
template <typename T>
__global__ void k_lowpass_divfree(C2<T>* v, Geom g) {
    const int n = g.n, nxh = n / 2;
    const size_t ps = plane_size(n);
    const size_t lidx = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (lidx >= size_t(n) * n * nxh) return;
    const size_t idx = sphys(n, lidx);
    const int kxi = lidx % nxh, kz = (lidx / nxh) % n, ky = lidx / (size_t(nxh) * n);
    const double kx = kxi * g.dkx, kyv = kwave(ky, n, g.dky), kzv = kwave(kz, n, g.dkz);
    const double k2 = kx * kx + kyv * kyv + kzv * kzv;
    C2<T> a[3];
    for (int c = 0; c < 3; c++) a[c] = v[c * ps + idx];
    if (k2 >= g.kM2) a[0] = a[1] = a[2] = mk<T>(T(0), T(0));
    if (k2 > 0) {
        const double ik2 = 1.0 / k2;  // as the step's projections
        const T t0 = T((kx * a[0].x + kyv * a[1].x + kzv * a[2].x) * ik2);
        const T t1 = T((kx * a[0].y + kyv * a[1].y + kzv * a[2].y) * ik2);
        a[0] = mk<T>(T(a[0].x - t0 * kx), T(a[0].y - t1 * kx));
        a[1] = mk<T>(T(a[1].x - t0 * kyv), T(a[1].y - t1 * kyv));
        a[2] = mk<T>(T(a[2].x - t0 * kzv), T(a[2].y - t1 * kzv));
    } else {
        a[0] = a[1] = a[2] = mk<T>(T(0), T(0));
    }
    for (int c = 0; c < 3; c++) v[c * ps + idx] = a[c];
}

// Biot-Savart into a spectral field (compute_velocity without symmetrize;
// the caller symmetrizes), used for host-visible cvelocity.
template <typename T>
__global__ void k_biot_savart(const C2<T>* __restrict__ w, C2<T>* __restrict__ u, Geom g) {
    const int n = g.n, nxh = n / 2;
    const size_t ps = plane_size(n);
    const size_t lidx = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (lidx >= size_t(n) * n * nxh) return;
    const size_t idx = sphys(n, lidx);
    const int kxi = lidx % nxh, kz = (lidx / nxh) % n, ky = lidx / (size_t(nxh) * n);
    const double kx = kxi * g.dkx, kyv = kwave(ky, n, g.dky), kzv = kwave(kz, n, g.dkz);
    const double k2 = kx * kx + kyv * kyv + kzv * kzv;
    const C2<T> a0 = w[idx], a1 = w[ps + idx], a2 = w[2 * ps + idx];
    if (k2 <= g.kM2 && k2 > 0) {
        const double ik2 = 1.0 / k2;  // as the step's fused Biot-Savart pass
        u[idx] = mk<T>(T(-(kyv * a2.y - kzv * a1.y) * ik2), T((kyv * a2.x - kzv * a1.x) * ik2));
        u[ps + idx] = mk<T>(T(-(kzv * a0.y - kx * a2.y) * ik2), T((kzv * a0.x - kx * a2.x) * ik2));
        u[2 * ps + idx] = mk<T>(T(-(kx * a1.y - kyv * a0.y) * ik2), T((kx * a1.x - kyv * a0.x) * ik2));
    } else {
        u[idx] = u[ps + idx] = u[2 * ps + idx] = mk<T>(T(0), T(0));
    }
}

// compute_vorticity (bfps/cpp/vorticity_equation.cpp:171-204): the curl
// w = i k x u for k^2 <= kM^2 (the k = 0 mode included), zero beyond; the
// caller symmetrizes.
template <typename T>
__global__ void k_curl(const C2<T>* __restrict__ u, C2<T>* __restrict__ w, Geom g) {
    const int n = g.n, nxh = n / 2;
    const size_t ps = plane_size(n);
    const size_t lidx = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (lidx >= size_t(n) * n * nxh) return;
    const size_t idx = sphys(n, lidx);
    const int kxi = lidx % nxh, kz = (lidx / nxh) % n, ky = lidx / (size_t(nxh) * n);
    const double kx = kxi * g.dkx, kyv = kwave(ky, n, g.dky), kzv = kwave(kz, n, g.dkz);
    const double k2 = kx * kx + kyv * kyv + kzv * kzv;
    const C2<T> a0 = u[idx], a1 = u[ps + idx], a2 = u[2 * ps + idx];
    if (k2 <= g.kM2) {
        w[idx] = mk<T>(T(-(kyv * a2.y - kzv * a1.y)), T(kyv * a2.x - kzv * a1.x));
        w[ps + idx] = mk<T>(T(-(kzv * a0.y - kx * a2.y)), T(kzv * a0.x - kx * a2.x));
        w[2 * ps + idx] = mk<T>(T(-(kx * a1.y - kyv * a0.y)), T(kx * a1.x - kyv * a0.x));
    } else {
        w[idx] = w[ps + idx] = w[2 * ps + idx] = mk<T>(T(0), T(0));
    }
}

// compute_gradient (bfps/cpp/field.cpp:1042-1101) of an ncs-component
// spectral field (ncs = 1 or 3): dst component j ncs + i = i k_j src_i for
// k^2 < kM^2 (strict), zero elsewhere.
template <typename T>
__global__ void k_gradient(const C2<T>* __restrict__ src, C2<T>* __restrict__ dst, Geom g, int ncs) {
    const int n = g.n, nxh = n / 2;
    const size_t ps = plane_size(n);
    const size_t lidx = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (lidx >= size_t(n) * n * nxh) return;
    const size_t idx = sphys(n, lidx);
    const int kxi = lidx % nxh, kz = (lidx / nxh) % n, ky = lidx / (size_t(nxh) * n);
    const double kv[3] = {kxi * g.dkx, kwave(ky, n, g.dky), kwave(kz, n, g.dkz)};
    const bool in = kv[0] * kv[0] + kv[1] * kv[1] + kv[2] * kv[2] < g.kM2;
    for (int i = 0; i < ncs; i++) {
        const C2<T> a = src[i * ps + idx];
        for (int j = 0; j < 3; j++)
            dst[(j * ncs + i) * ps + idx] = in ? mk<T>(T(-kv[j] * a.y), T(kv[j] * a.x)) : mk<T>(T(0), T(0));
    }
}

// kspace::cospectrum (bfps/cpp/kspace.cpp:521-598): FP64 shell sums
// S[s][i][j] += nxmodes (Re a_i Re b_j + Im a_i Im b_j), s = int(|k| / dk),
// k^2 <= kM^2, nxmodes = 1 at kx = 0 else 2.
template <typename T>
__global__ void k_cospectrum(const C2<T>* __restrict__ a, const C2<T>* __restrict__ bb, double* out,
                             Geom g, double dk, int nshells) {
    extern __shared__ double acc[];
    const int n = g.n, nxh = n / 2;
    const size_t ps = plane_size(n), nlog = size_t(n) * n * nxh;
    for (int i = threadIdx.x; i < nshells * 9; i += blockDim.x) acc[i] = 0.0;
    __syncthreads();
    for (size_t lidx = size_t(blockIdx.x) * blockDim.x + threadIdx.x; lidx < nlog; lidx += size_t(gridDim.x) * blockDim.x) {
        const int kxi = lidx % nxh, kz = (lidx / nxh) % n, ky = lidx / (size_t(nxh) * n);
        const size_t idx = sphys(n, lidx);
        const double kx = kxi * g.dkx, kyv = kwave(ky, n, g.dky), kzv = kwave(kz, n, g.dkz);
        const double k2 = kx * kx + kyv * kyv + kzv * kzv;
        if (k2 > g.kM2) continue;
        const double nxm = kxi == 0 ? 1.0 : 2.0;
        const int s = int(sqrt(k2) / dk) * 9;
        C2<T> av[3], bv[3];
        for (int c = 0; c < 3; c++) { av[c] = a[c * ps + idx]; bv[c] = bb[c * ps + idx]; }
        for (int i = 0; i < 3; i++)
            for (int j = 0; j < 3; j++)
                atomicAdd(&acc[s + i * 3 + j], nxm * (double(av[i].x) * double(bv[j].x) + double(av[i].y) * double(bv[j].y)));
    }
    __syncthreads();
    for (int i = threadIdx.x; i < nshells * 9; i += blockDim.x)
        if (acc[i] != 0.0) atomicAdd(&out[i], acc[i]);
}

}  // namespace bfpsh

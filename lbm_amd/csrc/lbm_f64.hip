// FP64 D2Q9 solver on the GPU, for measuring the error of the f32 and
// FP16-shifted grids at sizes a CPU FP64 solver cannot reach in time.
//
// It is the textbook scheme (BGK collide of every cell with
// feq_k = w_k rho (1 + 3 c.u + 4.5 (c.u)^2 - 1.5 u.u), then a pull stream
// with half-way bounce-back) with the reference step's boundary rules
// (lbm-wgpu rewritten_shaders/stream/{e_w,n_s,ne_sw,se_nw}_stream.wgsl:31-62):
// a cell is streamed only if it is fluid, x != 0 and y < ny - 1; column 0
// holds the inflow equilibrium feq(1, (u_in, 0)); an upstream cell that is
// solid or outside the grid bounces back; the outlet's west-moving upstream is
// the next row's column 0 (reference mode) or x clamped to nx - 1
// (zero-gradient).  Every operation is written in the order of the textbook
// solver the tests compare it with, in IEEE double without contraction, so the
// two agree bit for bit.  No reference counterpart: the reference is f32 only.
//
// Layout: nine dense planes per state (element (k, x, y) at k * nx * ny +
// y * nx + x), a pre-collision state f and a post-collision scratch g.

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <new>
#include <string>
#include <vector>

#include "../../include/lbm_hip.h"
#include "staging.h"
#include "tile.h"

namespace {

// sum + c v for c = -1, 0, 1 (0 v is exact: the fused form has the bits of the
// two operations, also where v is not finite)
template <int c>
__device__ __forceinline__ double plus(double sum, double v) {
    return c == 0 ? fma(0.0, v, sum) : c > 0 ? sum + v : sum - v;
}

// jx / rho and jy / rho, each correctly rounded: as velocity() in d2q9.h, with
// the second Newton step on the reciprocal that a double takes before the
// quotient's residual (12 instead of 22 instructions, one reciprocal instead of
// two, four for the test).  The residual is exact for numerators down to
// 2^-900; a smaller quotient changes no bit of the collision's sums.  Against the
// plain divisions 20.8 -> 20.3 us a step at 2048 x 1024, 3.9 -> 3.6 at 640 x 320.
__device__ __forceinline__ void velocity64(double jx, double jy, double rho, double &ux, double &uy) {
    const double top = fmax(fmax(fabs(jx), fabs(jy)), fabs(rho));
    if (__builtin_expect(__all(rho >= 0x1p-20 && top <= 0x1p20), 1)) {
        double r = __builtin_amdgcn_rcp(rho);
        r = fma(fma(-rho, r, 1.0), r, r);
        r = fma(fma(-rho, r, 1.0), r, r);
        ux = jx * r;
        ux = fma(fma(-rho, ux, jx), r, ux);
        uy = jy * r;
        uy = fma(fma(-rho, uy, jy), r, uy);
        return;
    }
    ux = jx / rho;
    uy = jy / rho;
}

// f := f + om (feq - f) of one cell, in the textbook solver's order.  c.u of
// opposite directions are each other's negatives, so their even term is the
// same and 1 + 3 c.u becomes 1 - 3 c.u with the same bits.
__device__ __forceinline__ void collide64(double fl[9], double om) {
    double rho = 0.0, jx = 0.0, jy = 0.0;
    [&]<int... K>(std::integer_sequence<int, K...>) {
        ((rho += fl[K], jx = plus<cx(K)>(jx, fl[K]), jy = plus<cy(K)>(jy, fl[K])), ...);
    }(std::make_integer_sequence<int, 9>());
    double ux, uy;
    velocity64(jx, jy, rho, ux, uy);
    const double uu15 = 1.5 * (ux * ux + uy * uy);
    const double rho36 = 1.0 / 36 * rho, rho9 = 1.0 / 9 * rho;
    auto relax = [&](int k, double wrho, double t) { fl[k] = fl[k] + om * (wrho * (t - uu15) - fl[k]); };
    auto pair = [&](int k, double wrho, double cu) {  // k and its opposite
        const double c3 = 3.0 * cu, even = 4.5 * cu * cu;
        relax(k, wrho, 1.0 + c3 + even);
        relax(opp(k), wrho, 1.0 - c3 + even);
    };
    pair(E, rho9, fma(0.0, uy, ux));
    pair(S, rho9, fma(0.0, ux, uy));
    pair(SE, rho36, ux + uy);
    pair(NE, rho36, ux - uy);
    // (c.u = 0 u: 1 + 3 c.u + 4.5 (c.u)^2 is 1, or NaN)
    relax(C, 4.0 / 9 * rho, 1.0 + fma(0.0, ux, 0.0 * uy));
}

struct Cell64 {
    double f[9];
};

// every cell alike (nine plane uploads took 7 of 8 ms to create 2048 x 1024)
__global__ void k64_fill(double *__restrict__ f, size_t n, Cell64 c) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
#pragma unroll
    for (int k = 0; k < 9; ++k) f[k * n + i] = c.f[k];
}

__global__ void k64_collide(const double *__restrict__ f, double *__restrict__ g, size_t n, double om) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double fl[9];
#pragma unroll
    for (int k = 0; k < 9; ++k) fl[k] = f[k * n + i];
    collide64(fl, om);
#pragma unroll
    for (int k = 0; k < 9; ++k) g[k * n + i] = fl[k];
}

// ---- the steps after the first collision: several per launch ----------------------
//
// Between two post-collision states a step is a pull and a collision; the
// call's last one is the pull alone.  As in tile.h a block owns a region of 64
// columns x (waves x M) rows, every population of a cell in registers: the
// first pull reads memory, the others take columns through lane shifts, rows
// inside a wave directly and the rows between two waves through LDS (one
// barrier a step).  Cells whose pulls leave the region turn invalid, one ring a
// step, so a region writes its inner cells, steps - 1 in from each edge.
//
// Column 0 and the last row, which the stream does not write, have the same
// post-collision value at every step: pulls from them read `fixed`, the state
// of the call's first collision, which the launches leave alone there (as they
// leave the solid cells, which nothing pulls from), whichever buffer is the
// source.  Lane X of a region in reference mode holds column 0 one row on, what
// the outlet's west-moving populations pull.
//
// A step a launch was bound by HBM (2048 x 1024: 65 us a step, 4.7 TB/s).  Here
// a step moves 37 bytes a cell (6 steps a launch, halo included) and takes about
// 130 FP64 instructions and 25 to shift and select, 1.5 times counting the
// halo: 20 us, of which either alone is about 15, as two blocks a CU overlap the
// one's loads with the other's steps in part.  Select instructions keep an
// unstreamed cell's value: a version of the steps without them for waves that
// hold none took 154 instead of 100 registers at three rows a wave, and with
// them the second block (37 against 21 us).
// a cell's bounced populations (bits as in d2q9.h), or kFixed: not streamed
constexpr uint32_t kFixed = 0x100u;

template <int MODE>
__global__ void k64_flags(const uint8_t *__restrict__ solid, uint16_t *__restrict__ flags, int X, int Y) {
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    const int y = blockIdx.y;
    if (x >= X) return;
    const size_t i = (size_t)y * X + x;
    uint32_t b = 0;
    if (x == 0 || y == Y - 1 || solid[i]) {
        b = kFixed;
    } else {
#pragma unroll
        for (int k = 0; k < 9; ++k) {
            if (k == C) continue;
            int ux, uy;
            upstream<MODE>(k, x, y, X, ux, uy);
            if (uy < 0 || uy >= Y || solid[(size_t)uy * X + ux]) b |= 1u << bit(k);
        }
    }
    flags[i] = (uint16_t)b;
}

struct Tile64Args {
    int steps;     // 1 .. kTileMaxSteps
    int nbx, nby;  // regions across and down
    int last;      // the call's last step is among them: f = the pulled state
};

template <int CX>
__device__ __forceinline__ double shift64(double v) {
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = from_west_east<CX>((uint32_t)b), hi = from_west_east<CX>((uint32_t)(b >> 32));
    return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}

template <int MODE, int M, int NW>
__global__ __launch_bounds__(64 * NW, NW / 2) void k64_tile(const double *__restrict__ src, double *__restrict__ dst,
                                                    const double *fixed, const uint16_t *__restrict__ flags, int X,
                                                    int Y, double om, Tile64Args a) {
    extern __shared__ double ex64[];
    constexpr bool wrap = MODE == LBM_BOUNDARY_REFERENCE;
    constexpr int rows = NW * M;
    const int L = xcd_remap(blockIdx.x, a.nbx * a.nby);
    const int by = L / a.nbx, bx = L - by * a.nbx;
    const int lane = (int)threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int h = a.steps - 1;
    const int x = bx * (64 - 2 * h) + lane;
    const int ry0 = w * M, y0 = by * (rows - 2 * h) - 1 + ry0;  // the wave's first row in the region, in the grid
    const size_t n = (size_t)X * Y;
    const bool virt = wrap && x == X, outlet = x == X - 1;
    const bool owner_x = (bx == 0 || lane >= h) && (bx == a.nbx - 1 || lane < 64 - h) && x < X;

    double cur[M][9];
    uint32_t kind[M];
    const int x0 = bx * (64 - 2 * h);
    const uint32_t col = (uint32_t)lane * 8;  // (a row's address is uniform: no address of a lane's own to keep)
    if (bx > 0 && x0 + 64 < X && y0 > 0 && y0 + M < Y - 1) {
        // every upstream cell is inside the grid and streamed, or solid and
        // bounced (an unstreamed cell here is solid: nothing reads its value)
#pragma unroll
        for (int j = 0; j < M; ++j) {
            const ptrdiff_t at = (ptrdiff_t)(y0 + j) * X + x0;
#pragma unroll
            for (int k = 0; k < 9; ++k)
                cur[j][k] = *(const double *)((const char *)(src + k * n + (at - cy(k) * X - cx(k))) + col);
            kind[j] = *(const uint16_t *)((const char *)(flags + at) + col / 4);
        }
    } else {
#pragma unroll
        for (int j = 0; j < M; ++j) {
            const int y = y0 + j;
            const bool in = x < X && y >= 0 && y < Y;
            kind[j] = in ? flags[(size_t)y * X + x] : kFixed;
            // an unstreamed cell keeps its value; past the grid nothing is read
            const bool keep = kind[j] == kFixed;
            const size_t own = virt ? (size_t)min(y + 1, Y - 1) * X : (size_t)min(max(y, 0), Y - 1) * X + min(x, X - 1);
#pragma unroll
            for (int k = 0; k < 9; ++k) {
                int ux, uy;
                upstream<MODE>(k, x, y, X, ux, uy);
                uy = min(max(uy, 0), Y - 1);  // (bounced where it is outside)
                const double *from = keep || ux <= 0 || uy == Y - 1 ? fixed : src;
                cur[j][k] = from[k * n + (keep ? own : (size_t)uy * X + ux)];
            }
        }
    }
    uint32_t live = 0;  // bit j: the row has streamed cells
    bool any_bounce = false;
#pragma unroll
    for (int j = 0; j < M; ++j) {
        if (!__all(kind[j] == kFixed)) live |= 1u << j;
        any_bounce = any_bounce || (kind[j] & 0xFFu) != 0;
    }
    any_bounce = __any(any_bounce);
    if (any_bounce)
#pragma unroll
        for (int j = 0; j < M; ++j) {
            if (!(kind[j] & 0xFFu)) continue;
            const ptrdiff_t at = (ptrdiff_t)(y0 + j) * X + x0;
#pragma unroll
            for (int k = 0; k < 9; ++k)
                if (k != C && ((kind[j] >> bit(k)) & 1u))
                    cur[j][k] = *(const double *)((const char *)(src + opp(k) * n + at) + col);
        }

    // does a later step or the store need step s (from 1) of row j, of any of the wave's rows?
    auto row_needed = [&](int s, int j) {
        return (by == 0 || ry0 + j >= s - 1) && (by == a.nby - 1 || ry0 + j < rows - (s - 1)) && ((live >> j) & 1u);
    };
    auto needed = [&](int s) {
        return (by == 0 || ry0 + M - 1 >= s - 1) && (by == a.nby - 1 || ry0 < rows - (s - 1)) && live;
    };
    if (!(a.last && a.steps == 1))
#pragma unroll
        for (int j = 0; j < M; ++j) {
            if (!row_needed(1, j)) continue;
            double f[9];
#pragma unroll
            for (int k = 0; k < 9; ++k) f[k] = cur[j][k];
            collide64(f, om);
#pragma unroll
            for (int k = 0; k < 9; ++k) cur[j][k] = kind[j] == kFixed ? cur[j][k] : f[k];
            __builtin_amdgcn_sched_barrier(0);
        }

    auto advance = [&]<bool COLLIDE>(int s) {
        double *e = ex64 + (size_t)(s & 1) * NW * 6 * 64;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            e[(w * 6 + i) * 64 + lane] = cur[0][i];              // NW, N, NE
            e[(w * 6 + 3 + i) * 64 + lane] = cur[M - 1][6 + i];  // SW, S, SE
        }
        __syncthreads();
        if (!needed(s)) return;
        double south[3], north[3];  // S-movers of the row above, N-movers of the row below the wave
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            south[i] = e[(max(w - 1, 0) * 6 + 3 + i) * 64 + lane];
            north[i] = e[(min(w + 1, NW - 1) * 6 + i) * 64 + lane];
        }
#pragma unroll
        for (int j = 0; j < M; ++j) {
            if (!row_needed(s, j)) {
#pragma unroll
                for (int i = 0; i < 3; ++i) south[i] = cur[j][6 + i];
                continue;
            }
            double p[9];
            [&]<int... K>(std::integer_sequence<int, K...>) {
                (
                    [&] {
                        const double v = cy(K) > 0   ? south[K >= 6 ? K - 6 : 0]
                                         : cy(K) < 0 ? (j + 1 < M ? cur[j + 1 < M ? j + 1 : j][K] : north[K < 3 ? K : 0])
                                                     : cur[j][K];
                        const double sh = shift64<cx(K)>(v);
                        p[K] = !wrap && cx(K) < 0 && outlet ? v : sh;
                    }(),
                    ...);
            }(std::make_integer_sequence<int, 9>());
            if (any_bounce) {
                // (opaque: the tests of every row are otherwise kept in 16 M
                // scalar registers over the steps)
                uint32_t kd = kind[j];
                asm volatile("" : "+v"(kd));
#pragma unroll
                for (int k = 0; k < 9; ++k)
                    if (k != C && ((kd >> bit(k)) & 1u)) p[k] = cur[j][opp(k)];
            }
#pragma unroll
            for (int i = 0; i < 3; ++i) south[i] = cur[j][6 + i];
            if constexpr (COLLIDE) collide64(p, om);
#pragma unroll
            for (int k = 0; k < 9; ++k) cur[j][k] = kind[j] == kFixed ? cur[j][k] : p[k];
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    const int collided = a.steps - (a.last ? 1 : 0);
    for (int s = 2; s <= collided; ++s) advance.template operator()<true>(s);
    if (a.last && a.steps > 1) advance.template operator()<false>(a.steps);

#pragma unroll
    for (int j = 0; j < M; ++j) {
        const int r = ry0 + j;
        const bool own = (by == 0 || r >= h) && (by == a.nby - 1 || r < rows - h) && y0 + j < Y;
        if (!(own && owner_x && kind[j] != kFixed)) continue;
        double *const row = dst + ((ptrdiff_t)(y0 + j) * X + x0);
#pragma unroll
        for (int k = 0; k < 9; ++k) *(double *)((char *)(row + k * n) + col) = cur[j][k];
        __builtin_amdgcn_sched_barrier(0);
    }
}

// rho, u = j / rho (uy north-positive, as the reference's uy field)
__global__ void k64_macro(const double *__restrict__ f, double *__restrict__ out, size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double r = 0.0, jx = 0.0, jy = 0.0;
#pragma unroll
    for (int k = 0; k < 9; ++k) {
        const double v = f[k * n + i];
        r += v;
        jx += cx(k) * v;
        jy += cy(k) * v;
    }
    out[i] = r;
    out[n + i] = jx / r;
    out[2 * n + i] = -jy / r;
}

struct HErr {
    hipError_t e;
    const char *what;
};
struct AErr {
    const char *msg;
};
#define H64(x)                                  \
    do {                                        \
        hipError_t e_ = (x);                    \
        if (e_ != hipSuccess) {                 \
            (void)hipGetLastError();            \
            throw HErr{e_, #x};                 \
        }                                       \
    } while (0)

thread_local std::string g_f64_error;

}  // namespace

struct lbm_f64 {
    int dev = 0;
    hipStream_t stream = nullptr;
    int X = 0, Y = 0, mode = 0;
    double omega = 1.0, u_in = 0.0;
    double *f = nullptr, *g = nullptr, *scratch = nullptr;
    uint8_t *solid = nullptr;
    uint16_t *flags = nullptr;
    uint64_t steps = 0;
    Staging staging;

    size_t n() const { return (size_t)X * Y; }
    void release() {
        (void)hipSetDevice(dev);
        staging.release();
        for (void *p : {(void *)f, (void *)g, (void *)scratch, (void *)solid})
            if (p) (void)hipFree(p);
        f = g = scratch = nullptr;
        solid = nullptr;
        flags = nullptr;
        if (stream) (void)hipStreamDestroy(stream);
        stream = nullptr;
    }
};

namespace {

template <class F>
int fguard(F &&fn) {
    try {
        fn();
        return LBM_OK;
    } catch (const HErr &e) {
        g_f64_error = std::string(e.what) + ": " + hipGetErrorString(e.e);
        return e.e == hipErrorOutOfMemory ? LBM_ENOMEM : LBM_EHIP;
    } catch (const HipError &e) {
        g_f64_error = std::string(e.what) + ": " + hipGetErrorString(e.e);
        return e.e == hipErrorOutOfMemory ? LBM_ENOMEM : LBM_EHIP;
    } catch (const AErr &e) {
        g_f64_error = e.msg;
        return LBM_EINVAL;
    } catch (const std::bad_alloc &) {
        g_f64_error = "host allocation failed";
        return LBM_ENOMEM;
    } catch (...) {
        g_f64_error = "unexpected exception";
        return LBM_EHIP;
    }
}

void fcheck(bool ok, const char *msg) {
    if (!ok) throw AErr{msg};
}

void flags64(lbm_f64 *h) {
    const dim3 grid((h->X + 255) / 256, h->Y);
    if (h->mode == LBM_BOUNDARY_REFERENCE)
        hipLaunchKernelGGL(k64_flags<LBM_BOUNDARY_REFERENCE>, grid, dim3(256), 0, h->stream, h->solid, h->flags, h->X,
                           h->Y);
    else
        hipLaunchKernelGGL(k64_flags<LBM_BOUNDARY_ZERO_GRADIENT>, grid, dim3(256), 0, h->stream, h->solid, h->flags,
                           h->X, h->Y);
    H64(hipGetLastError());
}

// one launch, from g to f or back
void tile64(lbm_f64 *h, int shape, int steps, bool to_f, bool last) {
    auto launch = [&]<int MODE, int SHAPE>() {
        constexpr TileShape sh = kTile64[SHAPE];
        constexpr auto kernel = &k64_tile<MODE, sh.m, sh.waves>;
        constexpr size_t lds = (size_t)sh.waves * 64 * 2 * 6 * sizeof(double);
        const Tile64Args a{steps, tile_nbx(h->X, steps), tile_nby(h->Y, sh.waves * sh.m, steps), last};
        tile_allow_lds<kernel>(lds, h->dev);
        hipLaunchKernelGGL(kernel, dim3(a.nbx * a.nby), dim3(64 * sh.waves), lds, h->stream, to_f ? h->g : h->f,
                           to_f ? h->f : h->g, h->g, h->flags, h->X, h->Y, h->omega, a);
    };
    auto shapes = [&]<int MODE>() {
        if (shape == 0) launch.template operator()<MODE, 0>();
        else if (shape == 1) launch.template operator()<MODE, 1>();
        else launch.template operator()<MODE, 2>();
    };
    if (h->mode == LBM_BOUNDARY_REFERENCE) shapes.template operator()<LBM_BOUNDARY_REFERENCE>();
    else shapes.template operator()<LBM_BOUNDARY_ZERO_GRADIENT>();
}

}  // namespace

extern "C" {

const char *lbm_f64_last_error(void) { return g_f64_error.c_str(); }

int lbm_f64_create(uint32_t nx, uint32_t ny, double omega, double u_in, int32_t boundary, int32_t device,
                   lbm_f64 **out) {
    return fguard([&] {
        fcheck(out != nullptr, "null output");
        *out = nullptr;
        fcheck(nx >= 3 && ny >= 3 && nx <= 65536 && ny <= 65535, "grid size out of range");
        fcheck(boundary == LBM_BOUNDARY_REFERENCE || boundary == LBM_BOUNDARY_ZERO_GRADIENT, "unknown boundary");
        H64(hipSetDevice(device));
        lbm_f64 *h = new lbm_f64();
        h->dev = device;
        h->X = (int)nx;
        h->Y = (int)ny;
        h->mode = boundary;
        h->omega = omega;
        h->u_in = u_in;
        try {
            H64(hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking));
            const size_t n = h->n();
            H64(hipMalloc(&h->f, 9 * n * sizeof(double)));
            H64(hipMalloc(&h->g, 9 * n * sizeof(double)));
            const size_t mask_bytes = (n + 255) / 256 * 256;  // the flags follow the mask
            H64(hipMalloc(&h->solid, mask_bytes + n * sizeof(uint16_t)));
            h->flags = (uint16_t *)(h->solid + mask_bytes);
            // walls on the first and last rows; everything at feq(1, (u_in, 0))
            std::vector<uint8_t> s(n, 0);
            for (uint32_t x = 0; x < nx; ++x) {
                s[x] = 1;
                s[(size_t)(ny - 1) * nx + x] = 1;
            }
            H64(hipMemcpy(h->solid, s.data(), n, hipMemcpyHostToDevice));
            flags64(h);
            Cell64 c;
            const double w[9] = {1.0 / 36, 1.0 / 9, 1.0 / 36, 1.0 / 9, 4.0 / 9, 1.0 / 9, 1.0 / 36, 1.0 / 9, 1.0 / 36};
            for (int k = 0; k < 9; ++k) {
                const double uu = u_in * u_in + 0.0 * 0.0;
                const double cu = cx(k) * u_in + 0.0;
                c.f[k] = w[k] * 1.0 * (1.0 + 3.0 * cu + 4.5 * cu * cu - 1.5 * uu);
            }
            hipLaunchKernelGGL(k64_fill, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, h->stream, h->f, n, c);
            H64(hipGetLastError());
            H64(hipStreamSynchronize(h->stream));
        } catch (...) {
            h->release();
            delete h;
            throw;
        }
        *out = h;
    });
}

int lbm_f64_destroy(lbm_f64 *h) {
    if (!h) return LBM_EINVAL;
    h->release();
    delete h;
    return LBM_OK;
}

int lbm_f64_set_mask(lbm_f64 *h, const uint8_t *solid) {
    return fguard([&] {
        fcheck(h && solid, "null argument");
        H64(hipSetDevice(h->dev));
        std::vector<uint8_t> s(solid, solid + h->n());
        for (auto &v : s) v = v == 1 ? 1 : 0;
        H64(hipMemcpyAsync(h->solid, s.data(), h->n(), hipMemcpyHostToDevice, h->stream));
        flags64(h);
        H64(hipStreamSynchronize(h->stream));
    });
}

int lbm_f64_step(lbm_f64 *h, uint32_t n) {
    return fguard([&] {
        fcheck(h != nullptr, "null handle");
        H64(hipSetDevice(h->dev));
        if (n == 0) return;
        const size_t cells = h->n();
        hipLaunchKernelGGL(k64_collide, dim3((unsigned)((cells + 255) / 256)), dim3(256), 0, h->stream, h->f, h->g,
                           cells, h->omega);
        const TilePlan plan = plan64(h->X, h->Y, n);
        const uint32_t low = n / plan.launches, more = n % plan.launches;
        for (uint32_t i = 0; i < plan.launches; ++i)
            tile64(h, plan.shape, (int)(low + (i < more)), i % 2 == 0, i + 1 == plan.launches);
        H64(hipGetLastError());
        h->steps += n;
    });
}

int lbm_f64_sync(lbm_f64 *h) {
    return fguard([&] {
        fcheck(h != nullptr, "null handle");
        H64(hipStreamSynchronize(h->stream));
    });
}

int lbm_f64_macro(lbm_f64 *h, double *rho, double *ux, double *uy) {
    return fguard([&] {
        fcheck(h != nullptr, "null handle");
        H64(hipSetDevice(h->dev));
        const size_t n = h->n();
        if (!h->scratch) H64(hipMalloc(&h->scratch, 3 * n * sizeof(double)));
        hipLaunchKernelGGL(k64_macro, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, h->stream, h->f, h->scratch,
                           n);
        H64(hipGetLastError());
        double *dst[3] = {rho, ux, uy};
        Piece p[3];
        int np = 0;
        for (int c = 0; c < 3; ++c)
            if (dst[c]) p[np++] = {dst[c], h->scratch + c * n, n * sizeof(double)};
        H64(h->staging.copy(h->dev, h->stream, p, np, true));
    });
}

int lbm_f64_read_f(lbm_f64 *h, double *f9) {
    return fguard([&] {
        fcheck(h && f9, "null argument");
        H64(hipSetDevice(h->dev));
        const Piece p{f9, h->f, 9 * h->n() * sizeof(double)};
        H64(h->staging.copy(h->dev, h->stream, &p, 1, true));
    });
}

int lbm_f64_step_count(const lbm_f64 *h, uint64_t *n) {
    if (!h || !n) return LBM_EINVAL;
    *n = h->steps;
    return LBM_OK;
}

}  // extern "C"

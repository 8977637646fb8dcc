// Several steps per launch for a tile of the grid that stays in registers,
// shared by the single grid (k_tile in lbm_grid.hip) and the batched engine.
#pragma once

#include <atomic>
#include <type_traits>

#include "lbm_common.h"
#include "tile_plan.h"

namespace {

// A block owns a region of 64 columns x (waves x M) rows: lane = column, a wave
// M consecutive rows, every population in registers.  The first of its `steps`
// steps reads A = C_n (pulled from memory; S-form: the cell's own state,
// collided only) and B (the other set, for the cells the stream does not
// write); the others pull from registers -- columns through DPP lane shifts,
// rows inside a wave directly, the rows between two waves through LDS (three
// populations each way, one barrier a step).  Cells whose pulls leave the
// region turn invalid, one ring a step, so a region of which steps - 1 cells on
// each side are halo writes its inner cells: A2 = C_{n+steps}, and B2 =
// C_{n+steps-1} where the next step reads it (the unstreamed cells) or, as the
// last launch of a call, everywhere, with the lagged moments of the last step.
//
// Cells that are not streamed (solid cells, column 0, the last row) take the
// moving populations of the set before the current one.  The reference outlet
// pulls from column 0 one row on, the flattened index: lane X of a region holds
// that column as cells of its own (row y: column 0 of row y + 1), and regions
// start one row above the grid, so that the outlet of row 0 finds column 0 of
// row 0 there.  The zero-gradient outlet pulls its own column.  Lanes and rows
// outside the grid carry values nothing reads: pulls from there are flagged as
// bounced.  Same per-cell operations as k_cell, so the same bits.
//
// What bounds it.  A step a launch was bound by HBM on large grids (385 us a
// step at 8192 x 4096 in f32) and by the launch on small ones (3.7 us at 400 x
// 160); two steps a launch from a ring of rows in LDS by its loads' latency and
// halo rows (265 us).  Here a step of a large grid moves 16 bytes a cell and the
// kernel is bound by VALU issue, 200 instructions a cell and step in f32, 171 in
// binary16 and 206 centred on the free stream, counting the halo, 1.4 times the
// cells (158, 134 and 155 us: the same time an instruction, not a byte), and a
// small grid by the 2 us a launch and the 1 us of a region's step (1.6 us a
// step).  More rows a wave mean less halo and fewer waves in flight: measured
// at 8192 x 4096 in f32, us per step of 6 steps a launch, for 2 x 16, 3 x 12 and
// 5 x 8 rows x waves: 176, 168, 188; binary16, of 5 steps, 2 x 16 (two blocks a
// CU, as its values need fewer registers) and 3 x 12: 141, 150.  3, 4, 6, 8
// steps a launch with 3 x 12 rows in f32: 246, 196, 168, 178.
struct TileArgs {
    int steps;         // 2 .. kTileMaxSteps
    int nbx, nby;      // regions across and down
    int sform, final;  // A is S_n; the call's last launch
};

constexpr size_t tile_lds(const TileShape &sh, size_t esize) {
    const size_t prev = sh.chain ? 8 * (size_t)(2 * sh.waves * sh.m + 64) : (size_t)sh.waves * sh.m * 8 * 64;
    return (size_t)sh.waves * 64 * 2 * 6 * sizeof(uint32_t) + prev * esize;
}

// a kernel's LDS above 64 KB has to be asked for, once per kernel and device
template <auto Kernel>
void tile_allow_lds(size_t lds, int dev) {
    static std::atomic<uint64_t> allowed{0};  // bit: device
    if (lds <= 65536) return;
    const uint64_t b = dev < 64 ? 1ull << dev : 0;
    if (b && (allowed.load(std::memory_order_relaxed) & b)) return;
    HIPCHK(hipFuncSetAttribute((const void *)Kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    allowed.fetch_or(b, std::memory_order_relaxed);
}

// lane - 1's (CX = 1) or lane + 1's (CX = -1) value; the end lanes keep their own
template <int CX, class V>
__device__ __forceinline__ V from_west_east(V v) {
    if constexpr (CX == 0) {
        return v;
    } else {
        const int i = __builtin_bit_cast(int, v);
        return __builtin_bit_cast(V, __builtin_amdgcn_update_dpp(i, i, CX > 0 ? 0x138 : 0x130, 0xF, 0xF, false));
    }
}

// The work of one block.  `ex`: tile_lds bytes of LDS.
template <class St, int MODE, int SHAPE>
__device__ __forceinline__ void tile_block(uint32_t *ex, const typename St::T *A, const typename St::T *B,
                                           typename St::T *__restrict__ A2, typename St::T *__restrict__ B2,
                                           const uint8_t *__restrict__ flags, const uint8_t *__restrict__ mask,
                                           const Geom &g, const TileArgs &a, int bx, int by, float *__restrict__ mom) {
    using T = typename St::T;
    using V = std::conditional_t<sizeof(T) == 2, uint32_t, T>;  // a stored value in a whole register
    constexpr bool wrap = MODE == LBM_BOUNDARY_REFERENCE;
    constexpr int M = tile_shape<T>(SHAPE).m, nw = tile_shape<T>(SHAPE).waves;
    constexpr bool chain = tile_shape<T>(SHAPE).chain;
    const int lane = (int)threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int h = a.steps - 1;
    constexpr int rows = nw * M;
    const int x = bx * (64 - 2 * h) + lane;
    const int ry0 = w * M, y0 = by * (rows - 2 * h) - 1 + ry0;  // the wave's first row in the region, in the grid
    const bool virt = wrap && x == g.X, outlet = x == g.X - 1;
    const bool owner_x = (bx == 0 || lane >= h) && (bx == a.nbx - 1 || lane < 64 - h) && x < g.X;
    // does a later step or the store need step s (from 1) of the wave's rows, of its row j?
    auto needed = [&](int s) {
        return (by == 0 || ry0 + M - 1 >= s - 1) && (by == a.nby - 1 || ry0 < rows - (s - 1)) && y0 < g.Y;
    };
    uint32_t live = 0;  // bit j: the row is in the grid and not all solid
    auto row_needed = [&](int s, int j) {
        return (by == 0 || ry0 + j >= s - 1) && (by == a.nby - 1 || ry0 + j < rows - (s - 1)) && ((live >> j) & 1u);
    };
    const uint32_t es = (uint32_t)sizeof(T), row_b = (uint32_t)(g.ys * es);
    // lane offsets of a row's columns x + 1, x, x - 1 (by the sign of c_x)
    const uint32_t col = (uint32_t)min(x, g.X - 1) * es;
    uint32_t off[3];
    off[0] = (uint32_t)min(x + 1, g.X - 1) * es;
    off[1] = col;
    off[2] = (uint32_t)min(max(x - 1, 0), g.X - 1) * es;
    const uint32_t own_col = virt ? 0u : col;  // column of the cell's own values

    V cur[M][9];
    // where an unstreamed cell's previous moving populations are, one every
    // `PS` elements (in registers they cost 8 M in every wave: 182 instead of 70
    // of them for M = 4)
    constexpr int PS = chain ? 2 * rows + 64 : 64;
    T *const prev0 = (T *)(ex + (size_t)2 * nw * 6 * 64);
    auto prev = [&](int j) {
        if constexpr (!chain) return prev0 + ((w * M + j) * 8 * 64 + lane);
        else return prev0 + (y0 + j == g.Y - 1 ? 2 * rows + lane : 2 * (ry0 + j) + (virt ? 1 : 0));
    };
    // a cell's bounced populations (the flag byte; of an unstreamed cell none),
    // kFixed: not streamed, kSolid: solid and, with `chain`, left out of the steps
    uint32_t kind[M];
    constexpr uint32_t kFixed = 0x100u, kSolid = 0x200u;
    bool any_fixed = false, any_bounce = false;

    auto base = [](const T *p, long long e) { return (const char *)(p + e); };
    auto load = [](const char *p, uint32_t o) { return (V) * (const T *)(p + o); };

    // ---- step 1 ----
#pragma unroll
    for (int j = 0; j < M; ++j) {
        const int y = y0 + j;
        kind[j] = 0;
        if (y >= g.Y) {  // uniform
#pragma unroll
            for (int k = 0; k < 9; ++k) cur[j][k] = V{};
            continue;
        }
        const int yc = max(y, 0);
        const char *mid = base(A, (long long)yc * g.ys), *dn = base(A, (long long)max(y - 1, 0) * g.ys),
                   *up = base(A, (long long)min(y + 1, g.Y - 1) * g.ys);
        // the cell's own row: column X's lane holds the next row's column 0
        const int yv = min(y + 1, g.Y - 1);
        const uint32_t own = virt ? (uint32_t)(yv - yc) * row_b : own_col;
        if (a.sform) {
#pragma unroll
            for (int k = 0; k < 9; ++k) cur[j][k] = load(mid + k * g.ks * es, own);
        } else {
#pragma unroll
            for (int k = 0; k < 9; ++k) {
                const char *row = cy(k) < 0 ? up : (cy(k) > 0 ? dn : mid);
                uint32_t o = off[cx(k) + 1];
                // the outlet's west-moving pulls: column 0 one row on (in row
                // 0 the row above is the clamped row 0 itself; past the last
                // row they are bounced, and read the row after the set)
                if (wrap && cx(k) < 0 && outlet) o = cy(k) > 0 && y < 1 ? 0u : row_b;
                if (k == C && virt) o = own;
                cur[j][k] = load(row + k * g.ks * es, o);
            }
        }
        uint32_t fl = 0;
        if (x < g.X && y >= 0) fl = flags[(size_t)y * g.pitch + x];
        if (virt) fl = kFixed;
        if (fl == kSlowCell) {
            const bool solid = mask[(size_t)y * g.pitch + x] == 1;
            if (chain && solid) fl = kSolid;
            else if (solid || x == 0 || y == g.Y - 1) fl = kFixed;
        }
        kind[j] = fl;
        if (!chain || !__all((fl & kSolid) != 0)) live |= 1u << j;
    }
#pragma unroll
    for (int j = 0; j < M; ++j) {
        any_fixed = any_fixed || (kind[j] & kFixed) != 0;
        any_bounce = any_bounce || (kind[j] & 0xFFu) != 0;
    }
    any_fixed = __any(any_fixed);
    any_bounce = __any(any_bounce);
    // own values of bounced and unstreamed cells, the other set's of unstreamed ones
    if (any_fixed || any_bounce) {
#pragma unroll
        for (int j = 0; j < M; ++j) {
            const int y = y0 + j;
            const bool fixed = (kind[j] & kFixed) != 0;
            if (!(fixed || ((kind[j] & 0xFFu) != 0 && !a.sform)) || y >= g.Y) continue;
            const int yc = max(y, 0);
            const uint32_t own = virt ? (uint32_t)(min(y + 1, g.Y - 1) - yc) * row_b : own_col;
            const char *ma = base(A, (long long)yc * g.ys), *mb = base(B, (long long)yc * g.ys);
            V o[9];
            if (!a.sform)
#pragma unroll
                for (int k = 0; k < 9; ++k)
                    if (k != C) o[k] = load(ma + k * g.ks * es, own);
            if (fixed) {
#pragma unroll
                for (int k = 0; k < 9; ++k) {
                    if (k == C) continue;
                    const V v = load(mb + k * g.ks * es, own);
                    prev(j)[bit(k) * PS] = (T)(a.sform ? v : o[k]);
                    if (!a.sform) cur[j][k] = v;
                }
            } else {
#pragma unroll
                for (int k = 0; k < 9; ++k)
                    if (k != C && ((kind[j] >> bit(k)) & 1u)) cur[j][k] = o[opp(k)];
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    if (needed(1)) {
#pragma unroll
        for (int j = 0; j < M; ++j) {
            if (!row_needed(1, j)) continue;
            float f[9];
            if (a.sform) {
#pragma unroll
                for (int k = 0; k < 9; ++k) f[k] = St::load((T)cur[j][k], k, g.sh);
            } else {
#pragma unroll
                for (int k = 0; k < 9; ++k)
                    f[k] = St::load_b((T)cur[j][k], k, k != C && ((kind[j] >> bit(k)) & 1u), g.sh);
            }
            St::collide(f, g.omega);
#pragma unroll
            for (int k = 0; k < 9; ++k) cur[j][k] = (V)St::store(f[k], k, g.sh);
            __builtin_amdgcn_sched_barrier(0);
        }
    }

    // one owned row of a set
    auto put = [&](T *dst, int j, const V(&v)[9]) {
        char *p = (char *)(dst + (long long)(y0 + j) * g.ys);
#pragma unroll
        for (int k = 0; k < 9; ++k) *(T *)(p + k * g.ks * es + col) = (T)v[k];
        __builtin_amdgcn_sched_barrier(0);
    };
    auto owned = [&](int j) {
        const int r = ry0 + j, y = y0 + j;
        return (by == 0 || r >= h) && (by == a.nby - 1 || r < rows - h) && y >= 0 && y < g.Y;
    };

    // ---- steps 2 .. steps ----  (FIXED: the wave holds unstreamed cells; every
    // wave passes the same barriers)
    auto advance = [&]<bool FIXED, bool LAST>(int s) {
        uint32_t *e = ex + (size_t)(s & 1) * nw * 6 * 64;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            e[(w * 6 + i) * 64 + lane] = __builtin_bit_cast(uint32_t, cur[0][i]);              // NW, N, NE
            e[(w * 6 + 3 + i) * 64 + lane] = __builtin_bit_cast(uint32_t, cur[M - 1][6 + i]);  // SW, S, SE
        }
        __syncthreads();
        if (!needed(s)) return;
        V south[3], north[3];  // S-movers of the row above, N-movers of the row below the wave
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            south[i] = __builtin_bit_cast(V, e[(max(w - 1, 0) * 6 + 3 + i) * 64 + lane]);
            north[i] = __builtin_bit_cast(V, e[(min(w + 1, nw - 1) * 6 + i) * 64 + lane]);
        }
#pragma unroll
        for (int j = 0; j < M; ++j) {
            if (!row_needed(s, j)) {
#pragma unroll
                for (int i = 0; i < 3; ++i) south[i] = cur[j][6 + i];
                continue;
            }
            V p[9];
            auto take = [&]<int K>() {
                const V v = cy(K) > 0 ? south[K - 6] : cy(K) < 0 ? (j + 1 < M ? cur[j + 1 < M ? j + 1 : j][K] : north[K])
                                                                 : cur[j][K];
                const V sh = from_west_east<cx(K)>(v);
                p[K] = !wrap && cx(K) < 0 && outlet ? v : sh;
            };
            take.template operator()<0>();
            take.template operator()<1>();
            take.template operator()<2>();
            take.template operator()<3>();
            p[C] = cur[j][C];
            take.template operator()<5>();
            take.template operator()<6>();
            take.template operator()<7>();
            take.template operator()<8>();
            float f[9];
#pragma unroll
            for (int k = 0; k < 9; ++k) f[k] = St::load((T)p[k], k, g.sh);
            if (any_bounce) {
                // (opaque: the tests of every row are otherwise kept in 16 M
                // scalar registers over the steps, and spilled)
                uint32_t kd = kind[j];
                asm volatile("" : "+v"(kd));
#pragma unroll
                for (int k = 0; k < 9; ++k)
                    if (k != C && ((kd >> bit(k)) & 1u)) f[k] = St::load((T)cur[j][opp(k)], opp(k), g.sh);
            }
            if constexpr (FIXED) {
                uint32_t kd = kind[j];
                asm volatile("" : "+v"(kd));
                if (kd & kFixed) {
                    T *const q = prev(j);
#pragma unroll
                    for (int k = 0; k < 9; ++k) {
                        if (k == C) continue;
                        f[k] = St::load(q[bit(k) * PS], k, g.sh);
                        q[bit(k) * PS] = (T)cur[j][k];
                    }
                }
            }
#pragma unroll
            for (int i = 0; i < 3; ++i) south[i] = cur[j][6 + i];
            const Moments m = St::collide(f, g.omega);
            if constexpr (LAST) {
                if (a.final && owned(j) && owner_x && !(kind[j] & kSolid)) {
                    const size_t i = (size_t)(y0 + j) * g.pitch + x;
                    mom[i] = m.jx;
                    mom[g.pstride + i] = m.jy;
                    mom[2 * g.pstride + i] = m.rho;
                }
            }
#pragma unroll
            for (int k = 0; k < 9; ++k) cur[j][k] = (V)St::store(f[k], k, g.sh);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto rest = [&]<bool FIXED>() {
        for (int s = 2; s < a.steps; ++s) advance.template operator()<FIXED, false>(s);
        if (a.final)  // C_{n+steps-1}: the other set after this call
#pragma unroll
            for (int j = 0; j < M; ++j)
            {
                if (owned(j) && owner_x && !(kind[j] & kSolid)) put(B2, j, cur[j]);
                __builtin_amdgcn_sched_barrier(0);
            }
        advance.template operator()<FIXED, true>(a.steps);
    };
    if (any_fixed) rest.template operator()<true>();
    else rest.template operator()<false>();

#pragma unroll
    for (int j = 0; j < M; ++j) {
        if (!(owned(j) && owner_x) || (kind[j] & kSolid)) continue;
        put(A2, j, cur[j]);
        if (!a.final && (kind[j] & kFixed)) {
            // (the rest population of the other set is never read)
            char *p = (char *)(B2 + (long long)(y0 + j) * g.ys);
#pragma unroll
            for (int k = 0; k < 9; ++k)
                if (k != C) *(T *)(p + k * g.ks * es + col) = prev(j)[bit(k) * PS];
        }
    }
    if constexpr (chain) {
        // the solid cells, each on its own
        for (int j = 0; j < M; ++j) {
            bool s = false;
#pragma unroll
            for (int i = 0; i < M; ++i) s = i == j ? (kind[i] & kSolid) != 0 : s;
            if (!(s && owner_x && owned(j))) continue;
            const char *pa = base(A, (long long)(y0 + j) * g.ys), *pb = base(B, (long long)(y0 + j) * g.ys);
            V c[9], q[9];
            float f[9];
#pragma unroll
            for (int k = 0; k < 9; ++k) {
                c[k] = load(pa + k * g.ks * es, col);
                q[k] = load(pb + k * g.ks * es, col);
            }
            Moments m;
            for (int i = 1; i <= a.steps; ++i) {
                const bool own = i == 1 && a.sform;  // S-form: the first step collides the cell's own state
#pragma unroll
                for (int k = 0; k < 9; ++k) f[k] = St::load((T)(own || k == C ? c[k] : q[k]), k, g.sh);
                // a cell whose two sets agree bit for bit and stay so under the
                // collision is the same after every step: solid cells soon are
                // (4096 x 2048 with 12% of the cells solid: 55 -> 52 us a step)
                bool still = true;
                m = St::collide(f, g.omega);
#pragma unroll
                for (int k = 0; k < 9; ++k) {
                    const V v = (V)St::store(f[k], k, g.sh);
                    still = still && __builtin_bit_cast(uint32_t, v) == __builtin_bit_cast(uint32_t, c[k]) &&
                            (k == C || __builtin_bit_cast(uint32_t, q[k]) == __builtin_bit_cast(uint32_t, c[k]));
                    q[k] = own && k != C ? q[k] : c[k];
                    c[k] = v;
                }
                if (__all(still)) break;
            }
            put(A2, j, c);
            put(B2, j, q);
            if (a.final) {
                const size_t i = (size_t)(y0 + j) * g.pitch + x;
                mom[i] = m.jx;
                mom[g.pstride + i] = m.jy;
                mom[2 * g.pstride + i] = m.rho;
            }
        }
    }
}

}  // namespace

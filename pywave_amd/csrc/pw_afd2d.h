// pw_afd2d.h -- several time steps of the 2D acoustic engine per launch (pw_afd.hip).
//
// fdm2d's step (pywave/src/wave_fdm.c:551-662) reads C_n and C_{n-1} and writes C_{n+1}; one step
// per launch moves 16 B a cell and, on grids of a few hundred cells a side, costs mostly the
// launch itself (3.3 us of which the memory traffic is a tenth).  Here a block advances its tile K
// steps: it loads the owned cells grown by 2K cells on every side (the stencil's reach per step is
// 2), keeps both levels and v^2 dt^2 of its cells in registers, publishes the current level in LDS
// once per step for the neighbours along z and across strips, and stores the last two levels to
// the other pair of fields (neighbour tiles still read the first pair).  Cells of the growth are
// recomputed by the tiles that share them, with the same operations in the same order, so the
// results are those of single steps bit for bit.  Lanes run along z (64 - 4K owned), each wave owns
// a strip of S columns, W waves make the tile; strips that no owned cell of a later step depends
// on stop computing.  Bound on small grids by the launch (about 3 us, spread over K steps) and the
// VALU and LDS latency of one tile's steps (0.8 us each): 161 x 161 takes 1.24 us a step against
// 2.92, 480 x 480 1.55 against 3.5.
#pragma once

#include <hip/hip_runtime.h>

namespace pw2d {

constexpr float kC0 = -30. / 12., kC1 = +16. / 12., kC2 = -1. / 12.;  // pywave/src/wave_fdm.c:15

// one shot's grid, fields and operands for the steps it, it + its, ... (nk of them)
struct Steps {
    const float *cur, *pv, *vv;  // C_n (damped), C_{n-1} (damped once), v^2 dt^2
    float *out_cur, *out_pv;     // C_{n+nk}, C_{n+nk-1}
    const float2 *fz, *fx;       // damping (lo, hi) per index; one of each pair is 1
    const int* src;              // 3*ns: gz, gx, - in padded coordinates
    const float* wav;            // ns*nt
    const float* tri;            // receiver data [nt][nx1] injected as sources, or null
    float* rec;                  // traces [nt][nx1] or null
    float* snap;                 // snapshots [nt/jsnap][nx1][nz1]
    int ns, nt, it, its, nk, jsnap;
    unsigned snaps;              // bit k: step k of the launch records a snapshot
    int nz, nx, nz2, nx2, ldz, nb, nz1, nx1;
    float idz, idx, cc;
};

template <int K, int S, int W>
struct Tile {
    static constexpr int halo = 2 * K, owned_z = 64 - 4 * K, cols = S * W, owned_x = cols - 4 * K;
};

// MANY: how a strip finds its sources.  With MANY strips look at the sources 64 at a time, one per
// lane; without, every strip of a tile that some source reaches goes through all of them, read as
// scalars.  The latter is faster for one source (161^2 cells, near the receivers' row, 1.34 against
// 1.37 us a step); with two it is slower (263 x 457 cells 1.65 against 1.46), with 100 and 1000 it takes
// 24.5 and 238 us against 2.0 and 6.5.
template <int K, int S, int W, bool MANY>
__device__ __forceinline__ void advance(const Steps& a, int tz, int tx)
{
    using T = Tile<K, S, W>;
    constexpr int H = T::halo, NX = T::cols;
    static_assert(K * S <= 64 && T::owned_z > 0 && T::owned_x > 0, "tile");
    __shared__ float lds[2][NX * 64 + 4];  // two cells of guard at either end
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int z0 = tz * T::owned_z - H, x0 = tx * T::owned_x - H;
    const int z = z0 + lane, c0 = w * S, xs = x0 + c0;
    const int L = a.ldz;
    const bool zact = z >= 0 && z < a.nz;
    const bool zin = zact && z >= 2 && z < a.nz2 - 2;
    // MANY: sources i0 .. i0 + 63, one per lane: their row, kFar where the stencil misses the strip.  The
    // first 64, loaded ahead of the fields, stay in registers over the launch.
    constexpr int kFar = -1;  // no source's: their stencils lie inside the grid
    auto near = [&](int i0, int& sx) -> int {
        const int i = i0 + lane;
        if (i >= a.ns) return kFar;
        const int sz = a.src[3 * i];
        sx = a.src[3 * i + 1];
        return sz >= z0 - 1 && sz <= z0 + 64 && sx >= xs - 1 && sx <= xs + S ? sz : kFar;
    };
    int sx0 = 0;
    const int sz0 = MANY ? near(0, sx0) : kFar;
    float u[S], p[S], vc[S], fx[S];
    unsigned lapmask[S];
    float fzz = 1.f;
    if (zact) {
        const float2 f = a.fz[z];
        fzz = f.x * f.y;  // one of the two is 1
    }
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const int x = xs + s;
        const bool xact = x >= 0 && x < a.nx;
        u[s] = p[s] = vc[s] = 0.f;
        fx[s] = 1.f;
        if (xact) {
            const float2 f = a.fx[x];
            fx[s] = f.x * f.y;
            if (zact) {
                const int j = x * L + z;
                u[s] = a.cur[j];
                p[s] = a.pv[j];
                vc[s] = a.vv[j];
            }
        }
        // zero on the Laplacian's rim and outside the updated domain, whose cells so stay zero
        lapmask[s] = zin && xact && x >= 2 && x < a.nx2 - 2 ? ~0u : 0u;
    }
    bool hit = false;  // some source's stencil reaches the strip (without MANY: the tile)
    if constexpr (MANY) {
        hit = __ballot(sz0 != kFar) != 0;
        for (int i0 = 64, sx; i0 < a.ns; i0 += 64) hit |= __ballot(near(i0, sx) != kFar) != 0;
    } else {
        for (int s = 0; s < a.ns; ++s)
            hit |= a.src[3 * s] >= z0 - 1 && a.src[3 * s] <= z0 + 64 && a.src[3 * s + 1] >= x0 - 1 && a.src[3 * s + 1] <= x0 + NX;
    }
    // the receiver row's lane, if the tile holds it; and if the tile owns it
    const int rlane = a.nb - z0;
    const bool rtile = rlane >= 0 && rlane < 64, rowned = rlane >= H && rlane < 64 - H;
    // the strip's receiver samples of every step, one per lane (time reversal)
    float tv = 0.f;
    if (a.tri && rtile && lane < K * S && lane / S < a.nk) {
        const int x = xs + lane % S - a.nb;
        if (x >= 0 && x < a.nx1) tv = a.tri[(size_t)(a.it + a.its * (lane / S)) * a.nx1 + x];
    }
    const bool zowned = zact && lane >= H && lane < 64 - H;
    int b = 0;
    for (int k = 0; k < a.nk; ++k) {
        const int t = a.it + a.its * k;
        const int lo = 2 * k, hi = NX - 2 * k;  // columns valid before this step
        float* row = lds[b] + 2;
        if (c0 + S > lo && c0 < hi) {
#pragma unroll
            for (int s = 0; s < S; ++s) row[(c0 + s) * 64 + lane] = u[s];
        }
        __syncthreads();
        b ^= 1;
        if (c0 + S <= lo + 2 || c0 >= hi - 2) continue;
        // the strip's columns and two on either side (the tile's edge strips read any column there:
        // what they compute from it is never used)
        float q[S + 4];
        const int cl = max(c0 - 2, 0), cr = min(c0 + S, NX - 2);
        q[0] = row[cl * 64 + lane];
        q[1] = row[(cl + 1) * 64 + lane];
        q[S + 2] = row[cr * 64 + lane];
        q[S + 3] = row[(cr + 1) * 64 + lane];
#pragma unroll
        for (int s = 0; s < S; ++s) q[s + 2] = u[s];
        float zn[S][4];
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const float* R = row + (c0 + s) * 64 + lane;
            zn[s][0] = R[-2]; zn[s][1] = R[-1]; zn[s][2] = R[1]; zn[s][3] = R[2];
        }
        __builtin_amdgcn_sched_barrier(0);  // every LDS read in flight before the first wait
        float nu[S];
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const float uc = q[s + 2];
            float lap = kC0 * uc * a.cc
                      + kC1 * (q[s + 1] + q[s + 3]) * a.idx
                      + kC2 * (q[s] + q[s + 4]) * a.idx
                      + kC1 * (zn[s][1] + zn[s][2]) * a.idz
                      + kC2 * (zn[s][0] + zn[s][3]) * a.idz;
            lap = __builtin_bit_cast(float, __builtin_bit_cast(unsigned, lap) & lapmask[s]);
            float pp = p[s];
            pp = pp * fzz; pp = pp * fx[s];
            float c = uc + (uc - pp);
            c = c + lap * vc[s];
            nu[s] = c;
        }
        if (hit) {  // in source order
            if constexpr (MANY) {
                for (int i0 = 0, sz = sz0, sx = sx0; i0 < a.ns; i0 += 64) {
                    if (i0) sz = near(i0, sx);
                    for (unsigned long long m = __ballot(sz != kFar); m; m &= m - 1) {
                        const int i = __builtin_ctzll(m);
                        const int dz = abs(z - __builtin_amdgcn_readlane(sz, i)), gx = __builtin_amdgcn_readlane(sx, i);
                        const float wv = a.wav[(size_t)(i0 + i) * a.nt + t];
#pragma unroll
                        for (int s = 0; s < S; ++s) {
                            const int dx = abs(xs + s - gx);
                            if (dx > 1) continue;
                            asm volatile("");  // a branch, not the quotients of every column and a select
                            if (dz <= 1) nu[s] = nu[s] + (vc[s] * wv) / (float)(dz + dx + 1);
                        }
                    }
                }
            } else {
                for (int i = 0; i < a.ns; ++i) {
                    const int dz = abs(z - a.src[3 * i]);
                    const float wv = a.wav[(size_t)i * a.nt + t];
#pragma unroll
                    for (int s = 0; s < S; ++s) {
                        const int dx = abs(xs + s - a.src[3 * i + 1]);
                        if (dz <= 1 && dx <= 1) nu[s] = nu[s] + (vc[s] * wv) / (float)(dz + dx + 1);
                    }
                }
            }
        }
        if (a.tri && rtile) {
#pragma unroll
            for (int s = 0; s < S; ++s) {
                const int x = xs + s - a.nb;
                if (x >= 0 && x < a.nx1) {
                    const float v = __shfl(tv, k * S + s);
                    if (lane == rlane) nu[s] = nu[s] + vc[s] * v;
                }
            }
        }
#pragma unroll
        for (int s = 0; s < S; ++s) {
            float c = nu[s];
            c = c * fzz; c = c * fx[s];
            p[s] = u[s];
            u[s] = c;
        }
        const bool snap = (a.snaps >> k) & 1;
        if ((a.rec && rowned) || snap) {
#pragma unroll
            for (int s = 0; s < S; ++s) {
                const int x = xs + s - a.nb;
                if (c0 + s < H || c0 + s >= NX - H || x < 0 || x >= a.nx1) continue;
                if (a.rec && lane == rlane && rowned) a.rec[(size_t)t * a.nx1 + x] = u[s];
                if (snap && zowned && z >= a.nb && z < a.nb + a.nz1)
                    a.snap[((size_t)(t / a.jsnap) * a.nx1 + x) * a.nz1 + (z - a.nb)] = u[s];
            }
        }
    }
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const int x = xs + s;
        if (zowned && c0 + s >= H && c0 + s < NX - H && x < a.nx) {
            const int j = x * L + z;
            a.out_cur[j] = u[s];
            a.out_pv[j] = p[s];
        }
    }
}

}  // namespace pw2d

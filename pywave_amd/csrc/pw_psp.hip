// pw_psp.hip -- the pseudo-spectral Laplacian of pywave's aps2d/aps3d on MI355X.
//
// Reference path (pywave = github.com/chenyk1990/pywave):
//   entry        pywave/aps2d.py:4-90, pywave/aps3d.py:4-94 -> apscfun (pywave/src/aps.c), whose set-up
//                is afd's; only the Laplacian of the time loop differs
//   engine       pywave/src/wave_psp.c:367-635 (psm2d), :25-365 (psm): wave = IFFT(-(2 pi |k|)^2 FFT(curr))
//   transforms   pywave/src/wave_fft2.c:72-151, wave_fft3.c:96-200 over the KISS FFT the reference
//                vendors (pywave/src/wave_kissfft.c)
//
// Each transform runs the KISS algorithm's arithmetic exactly, laid out for the GPU.  The recursive
// decimation of KISS becomes a digit-reversed read followed by one butterfly pass per factorisation
// level, deepest first.  All butterflies of a level are independent and each computes what KISS's
// radix-2/3/4/5 butterfly computes for its index (same twiddles, same f32 operation order), so
// every wavenumber and every output sample is bit-identical to the reference's.  Two neighbouring
// levels of radices p1, p2 (p1 p2 <= 16) run as one pass: a thread holds the p1 p2 elements they
// mix in registers, so a 144-point line (4 4 3 3) passes through LDS once instead of four times.
// The first pass of a line along x or y reads its elements from global memory in digit-reversed
// order, the last one writes global memory; lanes run over neighbouring lines, so both move whole
// 128 B segments and LDS accesses ([element][line]) are free of bank conflicts.  The real
// transforms along z pack pairs of samples into a half-length complex transform and split it with
// KISS's super-twiddles.  Launches per time step: x forward, y (forward, wavenumber multiply,
// inverse; in 2D the x lines do this), x inverse, and one kernel that holds whole z columns: split
// and inverse transform, the leapfrog update of its cells, and the new field's forward transform,
// so the spectral Laplacian and the new field are never re-read from memory.
//
// Measured on the 144^3 grid (141^3 updated, 73 bins along z), us per launch under the tracer: x forward
// 8.8, y 16.0, x inverse 12.3, z columns 26.3; a step of a run 61, against 131 in six launches with one
// pass per level, all transforms through LDS and the bins at a stride of 73.  Half of that came from the stride:
// with 73 bins every 128 B segment of a 16-line load straddles two cache lines (a plain copy in
// this order 12.8 us per 25 MB, 5.4 us at a stride of 80).  Bound now: about 72 MB a step through
// the z kernel and 27 MB through each line pass, at 3 to 4 TB/s with the launch's ramp; on small 2D
// grids (17 us against 37 for 192 x 240) the chain of latencies of a line's passes.
#include <algorithm>
#include <cmath>
#include <string>
#include <vector>

#include <hip/hip_ext.h>

#include "pw_internal.h"

namespace {

struct cf {
    float r, i;
};

__device__ __forceinline__ cf cmul(cf a, cf b) { return {a.r * b.r - a.i * b.i, a.r * b.i + a.i * b.r}; }
__device__ __forceinline__ cf cadd(cf a, cf b) { return {a.r + b.r, a.i + b.i}; }
__device__ __forceinline__ cf csub(cf a, cf b) { return {a.r - b.r, a.i - b.i}; }

constexpr int kMaxPass = 12;
constexpr int kPairMax = 16;  // elements of a two-level pass (registers: 25 would halve the occupancy)

// one pass: levels of radix po (outer; 1: none) and pi (inner), inner stride m, twiddle steps; s:
// groups of the first pass within one inner stride
struct FftPass {
    int code;      // 10 po + pi
    int m, fo, fi, s, pi;
    float rm, rs, rpi;  // 1/m, 1/s, 1/pi
};

// one transform length; inverse transforms use the conjugate twiddles
struct FftDev {
    int n, npass;
    FftPass ps[kMaxPass];  // in running order, deepest levels first
    const cf* tw;          // n twiddles exp(-2 pi i k/n)
};

// A kernel whose first parameter is a FftDev reads it in place, from the kernel-argument segment in
// the constant address space: an ordinary by-value parameter indexed at run time in more than one
// place is copied to private memory (measured: the z kernel 26 -> 64 us per launch).
using Fft = const __attribute__((address_space(4))) FftDev*;
using FftPassC = const __attribute__((address_space(4))) FftPass;
__device__ __forceinline__ Fft fft_arg() { return (Fft)__builtin_amdgcn_kernarg_segment_ptr(); }

// a / b for 0 <= a < 2^22 and b >= 1 through the f32 reciprocal rb = 1/b (the product is within
// one of the quotient; one correction step each way)
__device__ __forceinline__ int qdiv(int a, int b, float rb)
{
    int q = (int)((float)a * rb);
    const int r = a - q * b;
    q += (r >= b) - (r < 0);
    return q;
}

// input element of the first element of the first pass's group c (digit reversal; computed, as a
// table in memory would put one more load in front of the line's)
__device__ __forceinline__ int first_input(Fft d, int c)
{
    int from = 0;
    for (int q = d->npass - 1; q > 0; --q) {
        FftPassC& ps = d->ps[q];
        const int e = qdiv(c, ps.s, ps.rs), jo = qdiv(e, ps.pi, ps.rpi);
        c -= e * ps.s;
        from += jo * ps.fo + (e - jo * ps.pi) * ps.fi;
    }
    return from;
}

// KISS's butterfly of radix P on v[0], v[S], ...: k the index within the level's stride, fs the
// level's twiddle step, n the transform length (the radix-3/5 constants sit at n/P)
template <int P, int S, bool INV>
__device__ __forceinline__ void butterfly(cf* v, int k, int fs, int n, const cf* tw)
{
    auto w = [&](int i) {
        cf t = tw[i];
        if (INV) t.i = -t.i;
        return t;
    };
    if constexpr (P == 2) {
        const cf t = cmul(v[S], w(k * fs));
        v[S] = csub(v[0], t);
        v[0] = cadd(v[0], t);
    } else if constexpr (P == 3) {
        const float ei = w(n / 3).i;
        const cf s1 = cmul(v[S], w(k * fs));
        const cf s2 = cmul(v[2 * S], w(2 * k * fs));
        const cf s3 = cadd(s1, s2);
        cf s0 = csub(s1, s2);
        const cf f0 = v[0];
        // KISS takes the half in double and rounds once; so does the FMA
        const cf fm = {__builtin_fmaf(-.5f, s3.r, f0.r), __builtin_fmaf(-.5f, s3.i, f0.i)};
        s0.r = s0.r * ei;
        s0.i = s0.i * ei;
        v[0] = cadd(f0, s3);
        v[2 * S] = {fm.r + s0.i, fm.i - s0.r};
        v[S] = {fm.r - s0.i, fm.i + s0.r};
    } else if constexpr (P == 4) {
        const cf s0 = cmul(v[S], w(k * fs));
        const cf s1 = cmul(v[2 * S], w(2 * k * fs));
        const cf s2 = cmul(v[3 * S], w(3 * k * fs));
        const cf f = v[0];
        const cf s5 = csub(f, s1), g = cadd(f, s1);
        const cf s3 = cadd(s0, s2), s4 = csub(s0, s2);
        v[2 * S] = csub(g, s3);
        v[0] = cadd(g, s3);
        const cf a = {s5.r + s4.i, s5.i - s4.r}, b = {s5.r - s4.i, s5.i + s4.r};
        v[S] = INV ? b : a;
        v[3 * S] = INV ? a : b;
    } else {
        const cf ya = w(n / 5), yb = w(2 * (n / 5));
        const cf s0 = v[0];
        const cf s1 = cmul(v[S], w(k * fs));
        const cf s2 = cmul(v[2 * S], w(2 * k * fs));
        const cf s3 = cmul(v[3 * S], w(3 * k * fs));
        const cf s4 = cmul(v[4 * S], w(4 * k * fs));
        const cf s7 = cadd(s1, s4), s10 = csub(s1, s4), s8 = cadd(s2, s3), s9 = csub(s2, s3);
        v[0] = {s0.r + (s7.r + s8.r), s0.i + (s7.i + s8.i)};
        const cf s5 = {s0.r + s7.r * ya.r + s8.r * yb.r, s0.i + s7.i * ya.r + s8.i * yb.r};
        const cf s6 = {s10.i * ya.i + s9.i * yb.i, -(s10.r * ya.i) - s9.r * yb.i};
        v[S] = csub(s5, s6);
        v[4 * S] = cadd(s5, s6);
        const cf s11 = {s0.r + s7.r * yb.r + s8.r * ya.r, s0.i + s7.i * yb.r + s8.i * ya.r};
        const cf s12 = {-(s10.i * yb.i) + s9.i * ya.i, s10.r * yb.i - s9.r * ya.i};
        v[2 * S] = cadd(s11, s12);
        v[3 * S] = csub(s11, s12);
    }
}

// one pass over a line's groups of PO*PI elements by the line's T threads: ld(base, jo, ji, pos)
// reads the element at position pos (group base, outer digit jo, inner digit ji), st(pos, v)
// stores it
template <int PO, int PI, bool INV, class LD, class ST>
__device__ __forceinline__ void pass_t(Fft d, int iq, const cf* tw, int t, int T, LD ld, ST st)
{
    FftPassC& q = d->ps[iq];
    const int n = d->n;
    const int m = q.m, ng = n / (PO * PI);
    for (int g = t; g < ng; g += T) {
        const int c = m > 1 ? qdiv(g, m, q.rm) : g, k = g - c * m;
        const int base = c * (PO * PI) * m + k;
        cf v[PO * PI];
        const int from = LD::reversed ? first_input(d, g) : 0;
#pragma unroll
        for (int jo = 0; jo < PO; ++jo)
#pragma unroll
            for (int ji = 0; ji < PI; ++ji) v[jo * PI + ji] = ld(from, jo * q.fo + ji * q.fi, base + (jo * PI + ji) * m);
#pragma unroll
        for (int jo = 0; jo < PO; ++jo) butterfly<PI, 1, INV>(v + jo * PI, k, q.fi, n, tw);
        if constexpr (PO > 1) {
#pragma unroll
            for (int ji = 0; ji < PI; ++ji) butterfly<PO, PI, INV>(v + ji, k + m * ji, q.fo, n, tw);
        }
#pragma unroll
        for (int e = 0; e < PO * PI; ++e) st(base + e * m, v[e]);
    }
}

template <bool INV, class LD, class ST>
__device__ __forceinline__ void run_pass(Fft d, int iq, const cf* tw, int t, int T, LD ld, ST st)
{
    switch (d->ps[iq].code) {
        case 44: pass_t<4, 4, INV>(d, iq, tw, t, T, ld, st); break;
        case 42: pass_t<4, 2, INV>(d, iq, tw, t, T, ld, st); break;
        case 43: pass_t<4, 3, INV>(d, iq, tw, t, T, ld, st); break;
        case 23: pass_t<2, 3, INV>(d, iq, tw, t, T, ld, st); break;
        case 25: pass_t<2, 5, INV>(d, iq, tw, t, T, ld, st); break;
        case 33: pass_t<3, 3, INV>(d, iq, tw, t, T, ld, st); break;
        case 35: pass_t<3, 5, INV>(d, iq, tw, t, T, ld, st); break;
        case 12: pass_t<1, 2, INV>(d, iq, tw, t, T, ld, st); break;
        case 13: pass_t<1, 3, INV>(d, iq, tw, t, T, ld, st); break;
        case 14: pass_t<1, 4, INV>(d, iq, tw, t, T, ld, st); break;
        default: pass_t<1, 5, INV>(d, iq, tw, t, T, ld, st); break;
    }
}

// element reads of a pass: in place from LDS, or in digit-reversed order from F (LDS or global)
struct LdsLine {
    const cf* F;
    int stride;
    static constexpr bool reversed = false;
    __device__ cf operator()(int, int, int pos) const { return F[pos * stride]; }
};
struct PermLine {
    const cf* F;
    int stride;
    bool on;  // lanes past the last line read nothing
    static constexpr bool reversed = true;
    __device__ cf operator()(int from, int off, int) const
    {
        return on ? F[(unsigned)((from + off) * stride)] : cf{0.f, 0.f};
    }
};

struct PsGeo {
    int n1, n2, n3, nk, h;  // padded z (real), x, y; nk = n1/2 + 1; h = n1/2
    int ldk;                // stride of the half spectrum's columns: nk rounded up to 16 (128 B)
    int ldp;                // and of its planes
    int ldz;
    long long ldxy;
    float wwt;              // 1/(n1 n2 n3)
};

// Complex transforms along x (stride ldk, n2 points) or y (stride ldp, n3 points), LPB
// neighbouring wavenumber lines (consecutive along z, adjacent in memory) per block, NT/LPB
// threads a line.  MODE 0: forward; 1: inverse; 2: forward, multiply by the wavenumber operator,
// inverse.
template <int MODE, int LPB, int NT>
__global__ __launch_bounds__(NT) void k_ps_line(FftDev arg, PsGeo g, cf* __restrict__ tmp, int axis,
                                                const float* __restrict__ lapl)
{
    const Fft d = fft_arg();
    extern __shared__ cf sh[];
    constexpr int T = NT / LPB;
    const int tid = threadIdx.x, l = tid % LPB, t = tid / LPB;
    const int ngrp = (g.nk + LPB - 1) / LPB;
    const int i10 = (blockIdx.x % ngrp) * LPB, o = blockIdx.x / ngrp;
    const bool on = i10 + l < g.nk;
    long long base;
    int stride;  // offsets within a line stay below 2^31 (ps_create)
    if (axis == 0) { base = (long long)o * g.ldp + i10; stride = g.ldk; }
    else { base = (long long)o * g.ldk + i10; stride = g.ldp; }
    const int n = d->n;
    cf* B = sh + l;  // this line, element stride LPB
    cf* tw = sh + n * LPB * (MODE == 2 ? 2 : 1);
    for (int i = tid; i < n; i += NT) tw[i] = d->tw[i];
    cf* line = tmp + base + l;
    // the operator's values for the multiply, loaded ahead of the transform
    constexpr int WL = 10;
    const float* lp = lapl + base + l;
    float w[MODE == 2 ? WL : 1];
    auto load_w = [&](int i0) {
#pragma unroll
        for (int j = 0; j < WL; ++j) w[j] = on && i0 + j * T < n ? lp[(unsigned)((i0 + j * T) * stride)] : 0.f;
    };
    if constexpr (MODE == 2) load_w(t);
    auto lds = [B](int pos, cf v) { B[pos * LPB] = v; };
    auto out = [line, stride, on](int pos, cf v) { if (on) line[(unsigned)(pos * stride)] = v; };
    constexpr bool I0 = MODE == 1;
    const LdsLine own{B, LPB};
    // (the first pass's twiddles are the same few for every thread: read from global memory, it
    // needs no barrier after their staging)
    run_pass<I0>(d, 0, d->tw, t, T, PermLine{line, stride, on}, lds);
    __syncthreads();
    const int mid = MODE == 2 ? d->npass : d->npass - 1;
    for (int q = 1; q < mid; ++q) {
        run_pass<I0>(d, q, tw, t, T, own, lds);
        __syncthreads();
    }
    if constexpr (MODE != 2) {
        if (d->npass > 1) run_pass<I0>(d, d->npass - 1, tw, t, T, own, out);
        else for (int i = t; i < n; i += T) out(i, B[i * LPB]);
    } else {
        // wavenumber multiply in place, then the inverse from the other line buffer
        for (int i0 = t; i0 < n; i0 += WL * T) {
            if (i0 > t) load_w(i0);
#pragma unroll
            for (int j = 0; j < WL; ++j)
                if (i0 + j * T < n) {
                    const cf a = B[(i0 + j * T) * LPB];
                    B[(i0 + j * T) * LPB] = {a.r * w[j], a.i * w[j]};
                }
        }
        __syncthreads();
        cf* C = B + n * LPB;
        auto ldc = [C](int pos, cf v) { C[pos * LPB] = v; };
        const LdsLine ownc{C, LPB};
        run_pass<true>(d, 0, tw, t, T, PermLine{B, LPB, true}, ldc);
        __syncthreads();
        for (int q = 1; q < d->npass - 1; ++q) {
            run_pass<true>(d, q, tw, t, T, ownc, ldc);
            __syncthreads();
        }
        if (d->npass > 1) run_pass<true>(d, d->npass - 1, tw, t, T, ownc, out);
        else for (int i = t; i < n; i += T) out(i, C[i * LPB]);
    }
}

constexpr int z_stride(int lpb) { return lpb > 1 ? lpb + 1 : 1; }

__device__ __forceinline__ float damp_axis(float v, float2 a) { return (v * a.x) * a.y; }

constexpr int kFew = 4, kNear = 256;  // sources a block looks at without listing them; sources it can list

// One time step of LPB neighbouring z columns (x0 .. x0+LPB-1 of plane y): split and half-length
// inverse transform of their bins, centering sign and 1/(n1 n2 n3) -> the spectral Laplacian of
// C_n; psm2d/psm's update of the columns' cells (pywave/src/wave_psp.c:518-581, :193-256):
// leapfrog, injection, damping of both levels, receivers and snapshots; then centering sign and
// real transform of the new columns -> tmp [n3][ldp: n2][ldk] for the next step.  inv = 0 skips to the
// forward transform of 'cur' (the first step's), fwd = 0 stops after the update (the last step).
// Lanes run along z for global accesses and over columns in the passes; LDS elements are
// LPB + 1 apart so both orders spread over the banks.
// MANY: more than kFew sources.
template <bool D3, int LPB, int NT, bool MANY>
__global__ __launch_bounds__(NT, LPB >= 8 ? 6 : 1) void k_ps_z(FftDev arg, PsGeo g, PsStep a, cf* __restrict__ tmp,
                                             const cf* __restrict__ sup, int inv, int fwd)
{
    const Fft d = fft_arg();
    extern __shared__ cf sh[];
    constexpr int T = NT / LPB, LD = z_stride(LPB);
    constexpr int PF = 5;  // cells of a thread whose operands are loaded together
    const int tid = threadIdx.x, h = g.h, nz = a.nz;
    const int x0 = blockIdx.x * LPB, y = blockIdx.y;
    const int l = tid % LPB, t = tid / LPB;   // line and thread of the passes
    const int c = tid / T, z0 = tid % T;      // column and lane of the global accesses
    const int x = x0 + c;
    const bool in_grid = x < g.n2;
    const bool upd = x < a.nx && y < a.ny;    // the column lies in the updated domain
    cf* A = sh;
    cf* B = sh + h * LD;
    cf* tw = sh + 2 * h * LD;
    cf* sp = tw + h;                        // super-twiddles
    float2* fz = (float2*)(sp + (h + 1) / 2);  // damping pairs along z
    for (int i = tid; i < h; i += NT) tw[i] = d->tw[i];
    for (int i = tid; i < h / 2; i += NT) sp[i] = sup[i];
    for (int i = tid; i < nz; i += NT) fz[i] = a.fz[i];
    // block-uniform bases, 32-bit lane offsets
    const long long f0 = (long long)y * g.ldxy + (long long)x0 * g.ldz;
    const float* __restrict__ cur = a.cur + f0;
    float* __restrict__ prev = a.pv + f0;
    const float* __restrict__ vv = a.vv + f0;
    cf* __restrict__ X = tmp + (long long)y * g.ldp + x0 * g.ldk;
    const unsigned col = (unsigned)c * g.ldz, xc = (unsigned)c * g.ldk;
    // The sources whose stencil reaches the block's columns, in source order: all of a few if one does;
    // of many, those that do, found by the first wave 64 at a time.  (With every cell of such a block
    // looking at all of 1000 sources a 2D step on 263 x 457 cells took 344 us, 31 with the list, 21 with
    // one source; the list, at hand for one source too, cost a 3D step 3 %.)
    __shared__ int near[MANY ? kNear + 1 : 1];  // their number, and which
    auto reach = [&](int s) {
        return abs(y - a.src[3 * s + 2]) <= 1 && a.src[3 * s + 1] >= x0 - 1 && a.src[3 * s + 1] <= x0 + LPB;
    };
    bool hit = false;
    if constexpr (!MANY) {
        for (int s = 0; s < a.ns; ++s) hit |= reach(s);
    } else if (tid < 64) {
        int n = 0;
        for (int s0 = 0; s0 < a.ns; s0 += 64) {
            const int s = s0 + tid;
            const bool on = s < a.ns && reach(s);
            const unsigned long long m = __ballot(on);
            const int k = n + __popcll(m & ((1ull << tid) - 1));
            if (on && k < kNear) near[1 + k] = s;
            n += __popcll(m);
        }
        if (tid == 0) near[0] = n;
    }
    const bool neg = g.n3 > 1 ? ((y & 1) != (x & 1)) : (x & 1);
    const float2 one = make_float2(1.f, 1.f);
    const float2 fxx = upd ? a.fx[x] : one, fyy = D3 && upd ? a.fy[y] : one;
    float pu[PF], pp[PF], pv[PF];
    auto load_cells = [&](int zb) {
#pragma unroll
        for (int j = 0; j < PF; ++j) {
            const int z = zb + j * T;
            const bool ok = upd && z < nz;
            pu[j] = ok ? cur[col + z] : 0.f;
            pp[j] = ok && inv ? prev[col + z] : 0.f;
            pv[j] = ok && inv ? vv[col + z] : 0.f;
        }
    };
    // few columns per block (small grids, registers to spare): the cells' operands are loaded ahead
    // of the transform; with many, their registers would cost waves
    if (LPB <= 4) load_cells(z0);
    float* Af = (float*)A;
    const float* Bf = (const float*)B;
    auto at = [c](int z) { return ((z >> 1) * LD + c) * 2 + (z & 1); };
    auto lds = [B, l](int pos, cf v) { B[pos * LD + l] = v; };
    const LdsLine own{B + l, LD};
    const PermLine first{A + l, LD, true};
    if (inv) {
        for (int k0 = z0; k0 <= h / 2; k0 += 4 * T) {
            cf xa[4], xb[4], xw[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int k = k0 + j * T;
                const bool ok = in_grid && k <= h / 2;
                xa[j] = ok ? X[xc + k] : cf{0.f, 0.f};
                xb[j] = ok ? X[xc + h - k] : cf{0.f, 0.f};
                xw[j] = ok && k > 0 ? sup[k - 1] : cf{0.f, 0.f};
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int k = k0 + j * T;
                if (k > h / 2) continue;
                if (k == 0) {
                    A[c] = {xa[j].r + xb[j].r, xa[j].r - xb[j].r};
                    continue;
                }
                cf w = xw[j];
                w.i = -w.i;  // the inverse's super-twiddles are the conjugates
                const cf fk = xa[j], fnkc = {xb[j].r, -xb[j].i};
                const cf fek = cadd(fk, fnkc), dd = csub(fk, fnkc);
                const cf fok = cmul(dd, w);
                const cf lo = cadd(fek, fok);
                cf hi = csub(fek, fok);
                hi.i = hi.i * -1.f;
                if (k != h - k) A[k * LD + c] = lo;
                A[(h - k) * LD + c] = hi;
            }
        }
        __syncthreads();
        run_pass<true>(d, 0, tw, t, T, first, lds);
        __syncthreads();
        for (int q = 1; q < d->npass; ++q) {
            run_pass<true>(d, q, tw, t, T, own, lds);
            __syncthreads();
        }
    }
    const int nby = D3 ? a.nb : 0;
    const bool model = x >= a.nb && x < a.nb + a.nx1 && y >= nby && y < nby + a.ny1;
    const long long r = (long long)(y - nby) * a.nx1 + (x - a.nb);
    const float w = neg ? -g.wwt : g.wwt;
    // (the list was published by the barriers of the inverse transform)
    const int listed = MANY && inv ? __builtin_amdgcn_readfirstlane(near[0]) : 0;
    const int nsrc = !MANY ? (hit ? a.ns : 0) : listed <= kNear ? listed : a.ns;
    auto cell = [&](int z, float u, float p, float vc) {
        const float2 fzz = fz[z];
        p = damp_axis(damp_axis(p, fzz), fxx);
        if (D3) p = damp_axis(p, fyy);
        float v = u + (u - p);
        v = v + (w * Bf[at(z)]) * vc;
        for (int i = 0; i < nsrc; ++i) {
            const int s = MANY && listed <= kNear ? __builtin_amdgcn_readfirstlane(near[1 + i]) : i;
            const int dz = abs(z - a.src[3 * s]), dx = abs(x - a.src[3 * s + 1]), dy = abs(y - a.src[3 * s + 2]);
            if (dz <= 1 && dx <= 1 && dy <= 1)
                v = v + (vc * a.wav[(size_t)s * a.nt + a.it]) / (float)(dz + dx + dy + 1);
        }
        const bool onrec = model && z == a.nb;
        if (a.tri && onrec) v = v + vc * a.tri[r];
        v = damp_axis(damp_axis(v, fzz), fxx);
        if (D3) v = damp_axis(v, fyy);
        prev[col + z] = v;
        if (a.rec && onrec) a.rec[r] = v;
        if (a.snap && model && z >= a.nb && z < a.nb + a.nz1) a.snap[r * a.nz1 + (z - a.nb)] = v;
        return v;
    };
    for (int zb = z0; zb < 2 * h; zb += PF * T) {
        if (LPB > 4 || zb > z0) load_cells(zb);
#pragma unroll
        for (int j = 0; j < PF; ++j) {
            const int z = zb + j * T;
            if (z < 2 * h) {
                float v = pu[j];
                if (inv && upd && z < nz) v = cell(z, pu[j], pp[j], pv[j]);
                Af[at(z)] = neg ? -v : v;
            }
        }
    }
    if (!fwd) return;
    __syncthreads();
    run_pass<false>(d, 0, tw, t, T, first, lds);
    __syncthreads();
    for (int q = 1; q < d->npass; ++q) {
        run_pass<false>(d, q, tw, t, T, own, lds);
        __syncthreads();
    }
    if (!in_grid) return;
    for (int k = z0; k <= h / 2; k += T) {
        if (k == 0) {
            const cf t0 = B[c];
            X[xc] = {t0.r + t0.i, 0.f};
            X[xc + h] = {t0.r - t0.i, 0.f};
            continue;
        }
        const cf fpk = B[k * LD + c], q = B[(h - k) * LD + c];
        const cf fpnk = {q.r, -q.i};
        const cf f1k = cadd(fpk, fpnk), f2k = csub(fpk, fpnk);
        const cf ww = cmul(f2k, sp[k - 1]);
        const cf lo = {(f1k.r + ww.r) * .5f, (f1k.i + ww.i) * .5f};
        const cf hi = {(f1k.r - ww.r) * .5f, (ww.i - f1k.i) * .5f};
        if (k != h - k) X[xc + k] = lo;  // at k == h-k the second store wins, as in KISS
        X[xc + h - k] = hi;
    }
}

// ---------------------------------------------------------------- host side
struct HostFft {
    std::vector<int> p, m, fs;  // level 0 = the top of KISS's recursion
    std::vector<cf> tw;
};

// KISS's factorisation (4 first, then 2, 3, 5, ...), the input strides of its recursion (fs) and
// its forward twiddles; false if a radix other than 2, 3, 4, 5 appears
bool host_fft(int n, HostFft& f)
{
    f.tw.resize(n);
    const double pi = 3.141592653589793238462643383279502884197169399375105820974944;
    for (int i = 0; i < n; ++i) {
        const double ph = -2 * pi * i / n;
        f.tw[i] = {(float)std::cos(ph), (float)std::sin(ph)};
    }
    int mm = n, pp = 4;
    const double fsq = std::floor(std::sqrt((double)mm));
    do {
        while (mm % pp) {
            pp = pp == 4 ? 2 : (pp == 2 ? 3 : pp + 2);
            if (pp > fsq) pp = mm;
        }
        mm /= pp;
        f.p.push_back(pp);
        f.m.push_back(mm);
    } while (mm > 1);
    for (int q : f.p)
        if (q != 2 && q != 3 && q != 4 && q != 5) return false;
    int fsacc = 1;
    for (int q : f.p) {
        f.fs.push_back(fsacc);
        fsacc *= q;
    }
    return true;
}

}  // namespace

struct PsLap {
    PsGeo g{};
    float* lapl = nullptr;
    cf* tmp = nullptr;
    std::vector<void*> bufs;
    FftDev z{}, x{}, y{};
    cf* sup = nullptr;
    int lz = 1, lx = 1, ly = 1;  // lines per block of the z, x and y kernels
};

namespace {

int upload(PsLap* P, const void* host, size_t bytes, void** dev)
{
    if (hipMalloc(dev, bytes ? bytes : 8) != hipSuccess) return PW_ERR_NOMEM;
    P->bufs.push_back(*dev);
    if (host && bytes && hipMemcpy(*dev, host, bytes, hipMemcpyHostToDevice) != hipSuccess) return PW_ERR_HIP;
    return PW_OK;
}

// pair: two levels per pass where their elements fit the registers
int make_dev(PsLap* P, int n, bool pair, FftDev& d, std::string& err)
{
    HostFft h;
    if (!host_fft(n, h)) {
        err = "spectral Laplacian: transform length " + std::to_string(n) + " has a prime factor above 5";
        return PW_ERR_ARG;
    }
    d = FftDev{};
    d.n = n;
    // passes from the deepest level up
    for (int L = (int)h.p.size() - 1; L >= 0;) {
        if (d.npass == kMaxPass) {
            err = "spectral Laplacian: too many factorisation levels";
            return PW_ERR_ARG;
        }
        FftPass& q = d.ps[d.npass++];
        const bool two = pair && L > 0 && h.p[L - 1] * h.p[L] <= kPairMax;
        q.code = 10 * (two ? h.p[L - 1] : 1) + h.p[L];
        q.m = h.m[L];
        q.rm = 1.f / (float)q.m;
        q.fi = h.fs[L];
        q.fo = two ? h.fs[L - 1] : 0;
        q.pi = h.p[L];
        q.rpi = 1.f / (float)q.pi;
        const FftPass& q0 = d.ps[0];
        q.s = std::max(1, q.m / (q0.code / 10 * q0.pi));
        q.rs = 1.f / (float)q.s;
        L -= two ? 2 : 1;
    }
    void* b = nullptr;
    const int rc = upload(P, h.tw.data(), h.tw.size() * sizeof(cf), &b);
    d.tw = (const cf*)b;
    return rc;
}

size_t line_lds(int n, int lpb, bool both) { return ((size_t)(both ? 2 : 1) * lpb + 1) * n * sizeof(cf); }
// k_ps_z: two line buffers, twiddles, super-twiddles, damping pairs
size_t z_lds(int h, int lpb) { return (((size_t)2 * z_stride(lpb) + 3) * h + (h + 1) / 2) * sizeof(cf); }

// A line or z column that has a block to itself gets 256 threads, a z column of more than kLongColumn
// pairs (whose LDS leaves at most three blocks on a CU) 512.  Measured, us a step with 64, 256 and
// 512 threads (two kernels of whole lines, 256 threads, before): 2D 181 x 227 cells 17.9, 17.2 and
// 16.9 (36.7), 960^2 65, 44 and 50 (56), 1760^2 214, 121 and 129 (164), 4560 x 160 124, 57 and 45
// (82); 3D 1560 x 160 x 160 1208, 761 and 937 (1342), 3060 x 90 x 90 1267, 671 and 609 (864).
constexpr int kLongColumn = 1200;

template <int MODE>
void launch_line(const PsLap* P, const FftDev& d, int axis, int lpb, int others, hipStream_t s)
{
    const PsGeo& g = P->g;
    const dim3 grid((unsigned)((g.nk + lpb - 1) / lpb * others));
    const size_t lds = line_lds(d.n, lpb, MODE == 2);
    if (lpb == 16) hipLaunchKernelGGL((k_ps_line<MODE, 16, 256>), grid, dim3(256), lds, s, d, g, P->tmp, axis, P->lapl);
    else if (lpb == 8) hipLaunchKernelGGL((k_ps_line<MODE, 8, 128>), grid, dim3(128), lds, s, d, g, P->tmp, axis, P->lapl);
    else if (lpb == 4) hipLaunchKernelGGL((k_ps_line<MODE, 4, 64>), grid, dim3(64), lds, s, d, g, P->tmp, axis, P->lapl);
    else hipLaunchKernelGGL((k_ps_line<MODE, 1, 256>), grid, dim3(256), lds, s, d, g, P->tmp, axis, P->lapl);
}

template <bool D3>
void launch_z(const PsLap* P, const PsStep& a, int inv, int fwd, hipStream_t s, hipEvent_t e0, hipEvent_t e1)
{
    const PsGeo& g = P->g;
    const int lpb = P->lz;
    const dim3 grid((unsigned)((g.n2 + lpb - 1) / lpb), (unsigned)g.n3);
    const size_t lds = z_lds(g.h, lpb);
#define PW_PSZ(LPB, NT)                                                                                       \
    do {                                                                                                      \
        if (a.ns > kFew)                                                                                      \
            hipExtLaunchKernelGGL((k_ps_z<D3, LPB, NT, true>), grid, dim3(NT), lds, s, e0, e1, 0, P->z, g, a, \
                                  P->tmp, P->sup, inv, fwd);                                                  \
        else                                                                                                  \
            hipExtLaunchKernelGGL((k_ps_z<D3, LPB, NT, false>), grid, dim3(NT), lds, s, e0, e1, 0, P->z, g,   \
                                  a, P->tmp, P->sup, inv, fwd);                                               \
    } while (0)
    if (lpb == 16) PW_PSZ(16, 256);
    else if (lpb == 8) PW_PSZ(8, 128);
    else if (lpb == 4) PW_PSZ(4, 64);
    else if (g.h > kLongColumn) PW_PSZ(1, 512);
    else PW_PSZ(1, 256);
#undef PW_PSZ
}

// Lines per block: 16 (128 B segments) where at least two blocks per CU remain and the buffers
// leave room for several blocks per CU, else fewer.  Measured, 16 against 8 and 4 lines along x and
// y and along z: 144^3 (141^3 updated) 61, 76 and 100 us a step, 120^3 40, 53 and 67 us; one line
// (64 threads) against four on the 2D 192 x 240 grid 17.9 against 20.5 (x) and 22.7 us (z).
int lines_per_block(long long lines, int others, size_t (*lds)(int, int), int n)
{
    for (int l : {16, 8, 4})
        if ((lines + l - 1) / l * others >= 512 && lds(n, l) <= 40 * 1024) return l;
    return 1;
}

}  // namespace

void ps_destroy(PsLap* P)
{
    if (!P) return;
    for (void* b : P->bufs)
        if (b) hipFree(b);
    delete P;
}

// the operator of psm2d/psm (pywave/src/wave_psp.c:115-126, :471-480): lapl = -k*k with
// k = 2 pi hypot(kx, kz) (3D: hypot(ky, hypot(kx, kz))) in double, kx = kx0 + ix dkx in f32 with
// centred x (and y) wavenumbers and kz >= 0
PsLap* ps_create(int n1, int n2, int n3, int ldz, long long ldxy, float dz, float dx, float dy, std::string& err)
{
    if (n1 < 2 || n1 % 2 || n2 < 1 || n3 < 1 || ldz < n1) {
        err = "spectral Laplacian: bad padded extents";
        return nullptr;
    }
    // z lines to 4680 samples, x and y lines to 1820 points: one line takes 24 B of LDS a point in
    // k_ps_line and 44 B a pair of samples in k_ps_z (103 KB at the longest)
    if (n1 > 4680 || std::max(n2, n3) > 1820) {
        err = "spectral Laplacian: transform lines may have up to 4680 samples along z and 1820 along x and y, not " +
              std::to_string(n1) + " x " + std::to_string(n2) + " x " + std::to_string(n3);
        return nullptr;
    }
    // 1/(n1 n2 n3) takes the cell count in int, and the lines' element offsets are 32-bit: below 2^31
    // cells there are fewer than 2^31 bins, the padding of the columns to 16 bins included (at most
    // 2^30 + 16 * 1820^2)
    if ((long long)n1 * n2 * n3 >= 1LL << 31) {
        err = "spectral Laplacian: the padded grid " + std::to_string(n1) + " x " + std::to_string(n2) + " x " +
              std::to_string(n3) + " holds 2^31 cells or more";
        return nullptr;
    }
    PsLap* P = new PsLap;
    PsGeo& g = P->g;
    g.n1 = n1; g.n2 = n2; g.n3 = n3; g.h = n1 / 2; g.nk = n1 / 2 + 1;
    g.ldk = (g.nk + 15) / 16 * 16;
    g.ldp = g.ldk * n2;
    g.ldz = ldz; g.ldxy = ldxy;
    g.wwt = 1.0 / (n1 * n2 * n3);
    const int nk = g.nk;
    std::vector<float> lapl((size_t)g.ldp * n3, 0.f);
    const double PI = 3.14159265358979323846264338328;
    const float dkz = 1. / (n1 * dz), dkx = 1. / (n2 * dx), kx0 = -0.5 / dx;
    const float dky = n3 > 1 ? (float)(1. / (n3 * dy)) : 0.f, ky0 = n3 > 1 ? (float)(-0.5 / dy) : 0.f;
    for (int iy = 0; iy < n3; ++iy) {
        const float ky = ky0 + iy * dky;
        for (int ix = 0; ix < n2; ++ix) {
            const float kx = kx0 + ix * dkx;
            for (int iz = 0; iz < nk; ++iz) {
                const float kz = 0.f + iz * dkz;
                const float k = n3 > 1 ? (float)(2 * PI * std::hypot((double)ky, std::hypot((double)kx, (double)kz)))
                                       : (float)(2 * PI * std::hypot((double)kx, (double)kz));
                lapl[(size_t)iy * g.ldp + ix * g.ldk + iz] = -k * k;
            }
        }
    }
    // super-twiddles of the real transforms (kiss_fftr_alloc)
    std::vector<cf> sf(std::max(1, g.h / 2));
    for (int i = 0; i < g.h / 2; ++i) {
        const double ph = -3.14159265358979323846264338327 * ((double)(i + 1) / g.h + .5);
        sf[i] = {(float)std::cos(ph), (float)std::sin(ph)};
    }
    void *a = nullptr, *b = nullptr, *t = nullptr;
    int rc = upload(P, lapl.data(), lapl.size() * 4, &a);
    if (!rc) rc = upload(P, sf.data(), sf.size() * sizeof(cf), &b);
    if (!rc) rc = upload(P, nullptr, (size_t)g.ldp * n3 * sizeof(cf), &t);
    P->lapl = (float*)a;
    P->sup = (cf*)b;
    P->tmp = (cf*)t;
    auto one = [](int n, int l) { return line_lds(n, l, false); };
    auto both = [](int n, int l) { return line_lds(n, l, true); };
    P->lz = lines_per_block(n2, n3, z_lds, g.h);
    P->lx = lines_per_block(nk, n3, n3 > 1 ? +one : +both, n2);
    P->ly = lines_per_block(nk, n2, both, n3);
    // A line that has a block of its own runs one level per pass: 60 threads of a 240-point line share
    // each pass, 16 would share a pair of levels (2D 181 x 227 step, 64 threads: 17.9 against 20.6 us).
    if (!rc) rc = make_dev(P, g.h, P->lz > 1, P->z, err);
    if (!rc) rc = make_dev(P, n2, P->lx > 1, P->x, err);
    if (!rc && n3 > 1) rc = make_dev(P, n3, P->ly > 1, P->y, err);
    if (rc) {
        if (err.empty()) err = "spectral Laplacian: device allocation failed";
        ps_destroy(P);
        return nullptr;
    }
    return P;
}

hipError_t ps_begin(PsLap* P, const PsStep& a, hipStream_t s)
{
    if (P->g.n3 > 1) launch_z<true>(P, a, 0, 1, s, nullptr, nullptr);
    else launch_z<false>(P, a, 0, 1, s, nullptr, nullptr);
    return hipGetLastError();
}

hipError_t ps_step(PsLap* P, const PsStep& a, bool last, hipStream_t s, hipEvent_t e0, hipEvent_t e1)
{
    const PsGeo& g = P->g;
    if (g.n3 == 1) {
        launch_line<2>(P, P->x, 0, P->lx, 1, s);
        launch_z<false>(P, a, 1, !last, s, e0, e1);
    } else {
        launch_line<0>(P, P->x, 0, P->lx, g.n3, s);
        launch_line<2>(P, P->y, 1, P->ly, g.n2, s);
        launch_line<1>(P, P->x, 0, P->lx, g.n3, s);
        launch_z<true>(P, a, 1, !last, s, e0, e1);
    }
    return hipGetLastError();
}

// Size-specialised FFT passes: every even length but 242 from 16 to 256 with primes up
// to 13, which is what a grid chosen for an FFT has (kernels and launchers;
// instantiated per precision and range of lengths in fft_fixed_f32_*.hip and
// fft_fixed_f64_*.hip).
//
// The length, the tile and the radices are compile-time, so all index
// arithmetic folds to shifts and constant multiplies.  The first DFT takes its
// inputs from HBM into registers and the last one writes straight back (column
// and complex row passes); between DFTs the elements cross LDS once.  Few
// large radices (two, where they fit) mean few crossings and barriers, which
// bound large FP32 fields; their registers and few threads bound FP64 and small
// fields.  So: three radices up to 6 where a length has them in FP64, and in
// FP32 up to 64 points; else two up to 20 in FP32, two or three up to 13 in
// FP64.  An evaluation, us: 144^3 FP64 205 with 12 12, 189 with 4 6 6; 64^3 FP64
// 59 with 8 8, 53 with 4 4 4; 64^3 FP32 45 and 43, 64 x 256 x 256 FP32 154 and
// 152, 256 x 256 x 64 FP32 158 and 161.  160^3, three spectra: FP32 x pass with
// the multiply 38 us with 8 4 5, 26 with 10 16; FP64 column passes take 126
// registers with 10 16 and 50 with 4 5 8 (33 us either way), the z C2R 37 and
// 33 us.  A length without passes of its own takes the generic kernels
// (fft.hip): 52 x 78 x 104, FP64, three spectra: y pass 29 us there, 4.5 here.
//
// Column passes address a flattened set of pencils c in [0, ncols): base(c) =
// (c / P) * Q + c % P, element stride S, which covers the y pass (P = nzc, Q =
// ny*nzc, S = nzc) and the x pass (P = Q = S = ny*nzc) without partial tiles
// at plane boundaries.
#pragma once
#include <algorithm>
#include <type_traits>

#include "dft.h"
#include "gspace.h"
#include "internal.h"
#include "pointwise.h"
#include "post.h"
#include "stream.h"

namespace ofdft {

struct Radices {
    int n = 0;  // number of DFTs, 0: no such split
    int r[3] = {1, 1, 1};
};
// two or three factors up to `most`, the largest as small and then the
// smallest as large as possible, in ascending order (the first DFT has the
// most threads, the last leaves the others idle)
constexpr Radices split(int n, int most) {
    Radices s{};
    for (int a = 2; a * a <= n; ++a)
        if (n % a == 0 && n / a <= most) {
            s.n = 2;
            s.r[0] = a;
            s.r[1] = n / a;
        }
    if (s.n) return s;
    int top = most + 1;
    for (int a = 2; a * a * a <= n; ++a)
        for (int b = a; a * b * b <= n; ++b) {
            const int c = n / (a * b);
            if (n % (a * b) == 0 && c <= top) {
                top = c;
                s.n = 3;
                s.r[0] = a;
                s.r[1] = b;
                s.r[2] = c;
            }
        }
    return s;
}

// the DFTs of length N; REV: in the opposite order
template <typename T, int N> struct SL {
    static constexpr bool small = (sizeof(T) == 8 || N <= 64) && split(N, 6).n == 3;
    // FP64: 14 where 13 leaves only a split from 2 (98, 154, 182)
    static constexpr int large = sizeof(T) == 4 ? 20 : (split(N, 13).r[0] > 2 ? 13 : 14);
    static constexpr int most = small ? 6 : large;
    static constexpr Radices s = split(N, most);
    static_assert(s.n >= 2, "length without a split");
    static constexpr int n = s.n;
    static constexpr int TP = N / s.r[0];  // threads per pencil
    template <bool REV, int I> static constexpr int rad() { return REV ? s.r[n - 1 - I] : s.r[I]; }
    static constexpr int first = s.r[0], last = s.r[n - 1];
};

// Which butterfly j of which pencil a thread takes in a DFT of NB butterflies
// per pencil, and where the pencil's elements are in LDS.  Columns: TILE
// adjacent pencils, the pencil fixed per thread (its column in HBM).  Rows:
// NPEN pencils LD apart, the butterflies of all pencils packed onto the first
// threads, so that a large radix leaves whole waves idle and not lanes of all.
template <int TILE> struct ColMap {
    static constexpr int STRIDE = TILE;
    template <int NB> struct At {
        int pen, j, base;
        bool act;
        __device__ __forceinline__ explicit At(int t) : pen(t % TILE), j(t / TILE), base(pen), act(j < NB) {}
    };
};
template <int NPEN, int LD> struct RowMap {
    static constexpr int STRIDE = 1;
    template <int NB> struct At {
        int pen, j, base;
        bool act;
        __device__ __forceinline__ explicit At(int t) : pen(t / NB), j(t - pen * NB), base(pen * LD), act(pen < NPEN) {}
    };
};

// DFT I and the ones after it, from the inputs v (elements j + r N / R of the
// thread's butterfly); done() gets the butterfly and outputs of the last one
// (elements j + r N / R again).  Twiddles w^(r k) from the LDS table.
template <typename T, int N, typename MAP, bool INV, bool REV, int I, int NS, typename C, int R, typename F>
__device__ __forceinline__ void dfts(C *buf, const C *tw, C (&v)[R], F &&done) {
    using L = SL<T, N>;
    const typename MAP::template At<N / R> m((int)threadIdx.x);
    if (m.act) {
        if constexpr (NS > 1) {
            const int k = m.j % NS;
#pragma unroll
            for (int r = 1; r < R; ++r) {
                C w = tw[r * k * (N / (NS * R))];
                if (INV) w.y = -w.y;
                v[r] = cmul(v[r], w);
            }
        }
        DFT<R, INV, C>::run(v);
    }
    if constexpr (I + 1 == L::n) {
        done(m, v);
    } else {
        if constexpr (I > 0) __syncthreads();  // everyone has read the last exchange
        if (m.act) {
            const int d = (m.j / NS) * NS * R + m.j % NS;
#pragma unroll
            for (int r = 0; r < R; ++r) buf[m.base + (d + r * NS) * MAP::STRIDE] = v[r];
        }
        __syncthreads();
        constexpr int R2 = L::template rad<REV, I + 1>();
        const typename MAP::template At<N / R2> m2((int)threadIdx.x);
        C u[R2];
        if (m2.act) {
#pragma unroll
            for (int r = 0; r < R2; ++r) u[r] = buf[m2.base + (m2.j + r * (N / R2)) * MAP::STRIDE];
        }
        dfts<T, N, MAP, INV, REV, I + 1, NS * R>(buf, tw, u, done);
    }
}

// runs of a batch that a launch leaves out: those whose entry of live (device
// memory, null: none) is 0
__device__ __forceinline__ bool run_off(const double *live, unsigned b) { return live != nullptr && live[b] == 0.0; }

// Consecutive workgroups go to the 8 XCDs in turn, each with its own L2.
// Contiguous tiles to one XCD: where a row of elements is no multiple of a
// cache line (the half grids' nzc = nz / 2 + 1), neighbouring tiles share lines.
__device__ __forceinline__ unsigned xcd_tile(unsigned b, unsigned n) {
    const unsigned q = n / 8, r = n % 8, x = b % 8;
    return x * q + min(x, r) + b / 8;
}

// ---------------------------------------------------------------- column pass
template <typename T, int N, int TILE, bool INV>
__global__ void __launch_bounds__((TILE *SL<T, N>::TP))
    k_cols_f(const cpx<T> *in, cpx<T> *out, long long bs, unsigned ncols, unsigned P, long long Q, long long S,
             unsigned vp, const cpx<T> *__restrict__ twg, T scale, const double *live, const double *gate) {
    if (gate_off(gate) || run_off(live, blockIdx.y)) return;
    using C = cpx<T>;
    constexpr int R = SL<T, N>::first, TP = SL<T, N>::TP;
    __shared__ C tw[N];
    __shared__ C buf[N * TILE];
    const int pen = threadIdx.x % TILE;
    const int j = threadIdx.x / TILE;
    const unsigned c = xcd_tile(blockIdx.x, gridDim.x) * TILE + pen;
    const unsigned row = c / P, cp = c - row * P;
    const bool valid = c < ncols && cp < vp;  // pad columns of a pitched layout are skipped
    const long long off = (long long)blockIdx.y * bs + (valid ? (long long)row * Q + cp : 0) + j * S;
    C v[R];
    const C *src = in + off;
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = valid ? src[r * TP * S] : C{(T)0, (T)0};
    for (int i = threadIdx.x; i < N; i += TILE * TP) tw[i] = twg[i];
    dfts<T, N, ColMap<TILE>, INV, false, 0, 1>(buf, tw, v, [&](auto &m, auto &u) {
        constexpr int RL = SL<T, N>::last;
        if (!valid || !m.act) return;
        C *dst = out + off;
#pragma unroll
        for (int r = 0; r < RL; ++r) dst[r * (N / RL) * S] = C{u[r].x * scale, u[r].y * scale};
    });
}

// The lengths that had passes of their own first.  Two things hold for them
// alone, as before the others got theirs: the device-driven TN accepts them
// (opt.hip), and FP32 half grids form the G-space factors of the evaluation in
// FP32 at these x lengths.  Every other FP32 pass with the multiply (full
// grids, the other lengths, the kinetic operator) forms and applies them in
// FP64, as the stand-alone multiply does.  An FP32 evaluation of 160^3: 167 us
// on the half grid, 178 on the full one; with FP32 factors 167 and 169.
constexpr bool first_length(int n) {
    for (int m : {32, 48, 64, 72, 80, 96, 100, 120, 128, 144, 160, 192, 200, 240, 256})
        if (n == m) return true;
    return false;
}

// G-space factors of the elements e = j, j + TP, ... of one (iy, iz) column,
// into fac[e * TILE], from |G|^2 of the column's fixed part plus fx * b1 in
// the factors' precision T.  Unrolled: around a loop the compiler keeps the
// constants of the FP64 functions in 100 registers more.
template <typename T, int N, int TP, int TILE>
__device__ __forceinline__ void xfactors(T *fac, const GParams &gp, int kind, int iy, int iz, int j, double tkf,
                                         double wtfac) {
    const int fy = ffreq(iy, gp.ny);
    // kinetic: the complex grid (fftfreq on all axes)
    const int fz = kind == 4 ? ffreq(iz, gp.nz) : (gp.full ? wrapf(iz, gp.nz) : iz);
    const double cx = fy * gp.B[3] + fz * gp.B[6], cy = fy * gp.B[4] + fz * gp.B[7], cz = fy * gp.B[5] + fz * gp.B[8];
    const bool yz0 = iy == 0 && iz == 0;
    const bool yznyq =
        gp.full && (((gp.ny & 1) == 0 && iy == gp.ny / 2) || ((gp.nz & 1) == 0 && iz == gp.nz / 2));
    auto each = [&](auto &&val) {
        const T bx = (T)gp.B[0], by = (T)gp.B[1], bz = (T)gp.B[2], dx = (T)cx, dy = (T)cy, dz = (T)cz;
#pragma unroll
        for (int i = 0; i < N / TP; ++i) {
            const int e = j + i * TP;
            const T fx = (T)ffreq(e, N);
            const T gx = fx * bx + dx, gy = fx * by + dy, gz = fx * bz + dz;
            T f = val(gx * gx + gy * gy + gz * gz, yz0 && e == 0);
            // a Nyquist point of a full grid: the mean with the alias partner
            if (kind != 4 && (yznyq || (gp.full && 2 * e == N)))
                f = (T)0.5 * (f + val((T)gsq(gp.B, wrapf(-ffreq(e, N), N), wrapf(-fy, gp.ny), wrapf(-fz, gp.nz)),
                                      false));
            fac[e * TILE] = f;
        }
    };
    const T sc = (T)gp.scale;
    if (kind == 0) {
        const T sig = (T)(gp.sigma * gp.sigma / 4.0);
        each([&](T gg, bool) {
            T f = (T)0.5 * gg * sc;
            if (gp.sigma > 0) f *= exp(-gg * sig);
            return f;
        });
    } else if (kind == 1) {
        const T itkf = (T)(1.0 / tkf), wsc = (T)(wtfac * gp.scale), lb = (T)gp.lbda;
        each([&](T gg, bool) { return lindhard_t<T>(fm::sqrt_n(gg) * itkf, lb, (T)1) * wsc; });
    } else if (kind == 2) {
        each([&](T gg, bool g0) { return g0 ? (T)0 : gdiv<T>((T)(4.0 * M_PI) * sc, gg); });
    } else if (kind == 3) {
        each([&](T gg, bool) { return (T)(radial_table(gp, sqrt((double)gg)) * gp.scale); });
    } else {
        // kinetic: 1/2 G^2 exp(-G^2 sigma^2 / 2)
        const T s2 = (T)(gp.sigma * gp.sigma / 2.0);
        each([&](T gg, bool) { return (T)0.5 * gg * exp(-gg * s2) * sc; });
    }
}

// x pass of the evaluation pipeline with the G-space multiply fused in:
// forward x transform, kernel value by spectrum slot, inverse x transform, in
// place.  With its radices in the opposite order, the inverse starts from the
// very elements a thread holds after the forward transform, so the multiply
// works on registers.  All threads make the factors (fewer hold spectrum
// elements after a large last radix) while the column loads are on their way,
// and hand them over in LDS.  FT: the precision of the factors and the product.
template <typename T, typename FT, int N, int TILE>
__global__ void __launch_bounds__((TILE *SL<T, N>::TP))
    k_xfused_f(cpx<T> *data, long long bs, unsigned ncols, unsigned pitch, unsigned vp,
               const cpx<T> *__restrict__ twg, GParams gp, const double *live, const double *gate) {
    if (gate_off(gate) || run_off(live, blockIdx.y)) return;
    using C = cpx<T>;
    constexpr int R = SL<T, N>::first, RL = SL<T, N>::last, TP = SL<T, N>::TP;
    __shared__ C tw[N];
    __shared__ C buf[N * TILE];
    __shared__ FT fac[N * TILE];
    const int pen = threadIdx.x % TILE;
    const int j = threadIdx.x / TILE;
    const unsigned c = blockIdx.x * TILE + pen;
    const unsigned iy = c / pitch, iz = c - iy * pitch;
    const bool valid = c < ncols && iz < vp;
    const long long S = ncols;  // x stride of the (nx, ny, pitch) layout
    C *col = data + (long long)blockIdx.y * bs + (valid ? c : 0) + j * S;
    C v[R];
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = valid ? col[r * TP * S] : C{(T)0, (T)0};
    for (int i = threadIdx.x; i < N; i += TILE * TP) tw[i] = twg[i];
    const int kind = gp.kind[gp.c2c ? 0 : blockIdx.y];
    double tkf = 1.0, wtfac = 1.0;
    if (kind == 1) wt_consts(gp, tkf, wtfac);
    if (valid) xfactors<FT, N, TP, TILE>(fac + pen, gp, kind, (int)iy, (int)iz, j, tkf, wtfac);
    C u[RL];
    dfts<T, N, ColMap<TILE>, false, false, 0, 1>(buf, tw, v, [&](auto &, auto &w) {
#pragma unroll
        for (int r = 0; r < RL; ++r) u[r] = w[r];
    });
    // the factors are in LDS since the first exchange's barrier
    if (j < N / RL) {
#pragma unroll
        for (int r = 0; r < RL; ++r) {
            const FT f = fac[(j + r * (N / RL)) * TILE + pen];
            u[r].x = (T)(u[r].x * f);
            u[r].y = (T)(u[r].y * f);
        }
    }
    __syncthreads();
    dfts<T, N, ColMap<TILE>, true, true, 0, 1>(buf, tw, u, [&](auto &, auto &w) {
        if (!valid) return;
#pragma unroll
        for (int r = 0; r < R; ++r) col[r * TP * S] = w[r];
    });
}

// ---------------------------------------------------------------- rows passes
// the transforms of NPEN pencils staged in LDS in natural order, back to
// natural order (between two barriers of the caller's)
template <typename T, int N, int NPEN, int LD, bool INV>
__device__ __forceinline__ void row_ffts(cpx<T> *buf, const cpx<T> *tw) {
    using C = cpx<T>;
    using MAP = RowMap<NPEN, LD>;
    constexpr int R = SL<T, N>::first, RL = SL<T, N>::last, TP = SL<T, N>::TP;
    const typename MAP::template At<TP> m((int)threadIdx.x);
    C v[R];
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = buf[m.base + m.j + r * TP];
    __syncthreads();
    dfts<T, N, MAP, INV, false, 0, 1>(buf, tw, v, [&](auto &ml, auto &u) {
        __syncthreads();
        if (ml.act) {
#pragma unroll
            for (int r = 0; r < RL; ++r) buf[ml.base + ml.j + r * (N / RL)] = u[r];
        }
    });
}

// Prologues of the NF spectra at a point x (and rho r for the linear-response
// ops).  AUX and B56 are fixed per launch (block-uniform branches select the
// instance), so the compiler never evaluates the linear-response cases or the
// general power speculatively for the element-wise ops that do not need them.
// Without AUX the linear-response codes (which need rho) cannot occur: the
// host rejects them.  In FP64 the square and cube roots of a point's spectra
// come from one inverse sixth root.
template <typename T, bool AUX, bool B56, int NF>
__device__ __forceinline__ void prologue_t(const int (&code)[NF], T x, T beta, T r, T (&out)[NF]) {
    const T base = AUX ? r : x;
    T sq = (T)0, cb = (T)0, rc = (T)0;  // of max(base, 1e-30) (sqrt: of base > 0)
    bool roots = false;
#pragma unroll
    for (int f = 0; f < NF; ++f) roots |= code[f] != OP_IDENTITY;
    if (roots) {
        rc = base < (T)1e-30 ? (T)1e-30 : base;
        if constexpr (std::is_same<T, double>::value) {
            const bool fin = rc < (double)INFINITY;
            const fm::SixthRoot s(base > 0.0 ? base : 1e-30);
            sq = fin ? s.sqrt() : rc;
            if constexpr (B56) cb = base < 1e-30 ? 1e-10 : (fin ? s.cbrt() : rc);
        } else {
            sq = fm::sqrt_c(base > (T)0 ? base : (T)1e-30);
            if constexpr (B56) cb = fm::cbrt(rc);
        }
    }
    const T sqc = base < (T)1e-30 ? (T)1e-15 : sq;  // sqrt(max(base, 1e-30))
#pragma unroll
    for (int f = 0; f < NF; ++f) {
        switch (code[f]) {
            case OP_SQRT_RHOM: out[f] = sq; break;
            case OP_POW_BETA:
                if constexpr (B56)
                    out[f] = sqc * cb;
                else
                    out[f] = fm::pow(rc, beta);
                break;
            case OP_DSQRT: out[f] = AUX ? fm::div(x, (T)2 * sq) : x; break;
            case OP_DPOW_BETA:
                if constexpr (AUX && B56)
                    out[f] = beta * fm::div(cb, sqc) * x;
                else if constexpr (AUX)
                    out[f] = beta * fm::pow(rc, beta - (T)1) * x;
                else
                    out[f] = x;
                break;
            default: out[f] = x;
        }
    }
}

// Rows R2C for NF spectra at once: NPEN packed pairs of rows per spectrum.
// The NF spectra transform the same input, each with its own prologue (NF = 1:
// spectrum blockIdx.y of inputs in_bs apart).  A thread's loads go out
// together, with row addresses clamped into the tile instead of branches (rows
// past the end are zeroed afterwards).  Output rows have pitch opitch >= N/2+1.
// partials[blockIdx.x] receives the FP64 sum of slot sum_slot over the tile.
template <typename T, int N, int NPEN, int NF>
__global__ void __launch_bounds__((NF *NPEN *SL<T, N>::TP))
    k_rows_r2c_f(const T *__restrict__ in, cpx<T> *__restrict__ out, long long in_bs, long long out_bs, long long nrows,
                 int opitch, const cpx<T> *__restrict__ twg, T scale, Prologue pro, double *partials,
                 int sum_slot, const double *gate) {
    if (gate_off(gate)) return;
    using C = cpx<T>;
    constexpr int TP = SL<T, N>::TP, LD = N + 1;
    constexpr int NT = NF * NPEN * TP;
    constexpr int ROWS = 2 * NPEN;
    constexpr int NZC = N / 2 + 1;
    __shared__ C tw[N];
    __shared__ C buf[NF * NPEN * LD];
    const int slot0 = blockIdx.y * NF;
    const T *src = in + slot0 * in_bs;
    const T *aux = reinterpret_cast<const T *>(pro.aux);
    const T *phi = reinterpret_cast<const T *>(pro.phi);
    const T beta = (T)pro.beta;
    const bool do_sum = partials != nullptr && sum_slot >= slot0 && sum_slot < slot0 + NF;
    int code[NF];
#pragma unroll
    for (int f = 0; f < NF; ++f) code[f] = pro.code[(slot0 + f) & 3];
    for (int i = threadIdx.x; i < N; i += NT) tw[i] = twg[i];
    double acc[1] = {0.0};
    const long long row0 = (long long)blockIdx.x * ROWS;
    const int nv = (int)min((long long)ROWS, nrows - row0);
    constexpr int NW = NPEN * N, PER = (NW + NT - 1) / NT;
    // point (pair, pos) of both rows: all loads of a thread go out together
    C x0[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int w = min((int)threadIdx.x + i * NT, NW - 1);
        const int p = w / N;
        const long long ea = (row0 + (2 * p < nv ? 2 * p : 0)) * N + (w - p * N);
        const long long eb = 2 * p + 1 < nv ? ea + N : ea;
        x0[i] = C{src[ea], src[eb]};
        if (phi) {
            const C f{phi[ea], phi[eb]};
            x0[i] = C{(T)(2.0 * (double)f.x * (double)x0[i].x), (T)(2.0 * (double)f.y * (double)x0[i].y)};
        }
    }
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int w = threadIdx.x + i * NT;
        if (NW % NT == 0 || w < NW) buf[w / N * LD + w % N] = x0[i];
    }
    // the prologues, each thread on its own points (unrolled only for the
    // fused spectra, where a thread has few)
    auto prep = [&](auto aux_c, auto b56_c) {
        constexpr bool AUX = decltype(aux_c)::value, B56 = decltype(b56_c)::value;
#pragma unroll NF == 3 ? PER : 1
        for (int i = 0; i < PER; ++i) {
            const int w = threadIdx.x + i * NT;
            if (NW % NT != 0 && w >= NW) break;
            const int p = w / N, pos = w - p * N;
            const bool la = 2 * p < nv, lb = 2 * p + 1 < nv;
            const C x = buf[p * LD + pos];
            C a{(T)0, (T)0};
            if constexpr (AUX) {
                const long long ea = (row0 + (la ? 2 * p : 0)) * N + pos;
                a = C{aux[ea], aux[lb ? ea + N : ea]};
            }
            T oa[NF], ob[NF];
            prologue_t<T, AUX, B56, NF>(code, x.x, beta, a.x, oa);
            prologue_t<T, AUX, B56, NF>(code, x.y, beta, a.y, ob);
            if (do_sum) acc[0] += (la ? (double)x.x : 0.0) + (lb ? (double)x.y : 0.0);
#pragma unroll
            for (int f = 0; f < NF; ++f)
                buf[(f * NPEN + p) * LD + pos] = C{la ? oa[f] : (T)0, lb ? ob[f] : (T)0};
        }
    };
    if (aux) {
        if (pro.b56)
            prep(std::true_type{}, std::true_type{});
        else
            prep(std::true_type{}, std::false_type{});
    } else {
        if (pro.b56)
            prep(std::false_type{}, std::true_type{});
        else
            prep(std::false_type{}, std::false_type{});
    }
    __syncthreads();
    row_ffts<T, N, NF * NPEN, LD, false>(buf, tw);
    __syncthreads();
    // separate the packed rows: A_k = (Z_k + conj Z_{N-k}) / 2, B_k = (Z_k - conj Z_{N-k}) / 2i
    for (int e = threadIdx.x; e < NF * NPEN * NZC; e += NT) {
        const int qq = e / NZC, k = e - qq * NZC;
        const int ff = qq / NPEN, pp = qq - ff * NPEN;
        const C z = buf[qq * LD + k];
        C zc = buf[qq * LD + (k == 0 ? 0 : N - k)];
        zc.y = -zc.y;
        C *o = out + (long long)(slot0 + ff) * out_bs + (row0 + 2 * pp) * opitch + k;
        if (2 * pp < nv) *o = C{(z.x + zc.x) * (T)0.5 * scale, (z.y + zc.y) * (T)0.5 * scale};
        if (2 * pp + 1 < nv) o[opitch] = C{(z.y - zc.y) * (T)0.5 * scale, -(z.x - zc.x) * (T)0.5 * scale};
    }
    if (do_sum) block_sums<1>(acc, partials);
}

// Rows C2R (irfft semantics: imaginary parts of k = 0 and Nyquist ignored).
// Each thread loads column k of a row pair (A of row 2p, B of row 2p+1) and
// stages A + iB at k and its Hermitian image conj(A) + i conj(B) at N - k of
// the packed pencil.  All loads of a tile are issued at once with clamped
// addresses.
template <typename T, int N, int NPEN>
__global__ void __launch_bounds__((NPEN *SL<T, N>::TP))
    k_rows_c2r_f(const cpx<T> *__restrict__ in, T *__restrict__ out, long long in_bs, long long out_bs,
                 long long nrows, int ipitch, const cpx<T> *__restrict__ twg, T scale, const double *gate) {
    if (gate_off(gate)) return;
    using C = cpx<T>;
    constexpr int TP = SL<T, N>::TP, LD = N + 1, NT = NPEN * TP, ROWS = 2 * NPEN;
    constexpr int NZC = N / 2 + 1, NW = NPEN * NZC, PER = (NW + NT - 1) / NT;
    __shared__ C tw[N];
    __shared__ C buf[NPEN * LD];
    const long long row0 = (long long)blockIdx.x * ROWS;
    const int nv = (int)min((long long)ROWS, nrows - row0);
    in += (long long)blockIdx.y * in_bs;
    T *dst = out + (long long)blockIdx.y * out_bs + row0 * N;
    C ra[PER], rb[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int w = min((int)threadIdx.x + i * NT, NW - 1);
        const int p = w / NZC, k = w - p * NZC;
        const C *a = in + (row0 + (2 * p < nv ? 2 * p : 0)) * ipitch + k;
        ra[i] = *a;
        rb[i] = a[2 * p + 1 < nv ? ipitch : 0];
    }
    for (int i = threadIdx.x; i < N; i += NT) tw[i] = twg[i];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int w = threadIdx.x + i * NT;
        if (NW % NT != 0 && w >= NW) continue;
        const int p = w / NZC, k = w - p * NZC;
        C a = ra[i], b = rb[i];
        if (k == 0 || 2 * k == N) a.y = b.y = (T)0;
        buf[p * LD + k] = C{a.x - b.y, a.y + b.x};
        if (k > 0 && 2 * k < N) buf[p * LD + N - k] = C{a.x + b.y, b.x - a.y};
    }
    __syncthreads();
    row_ffts<T, N, NPEN, LD, true>(buf, tw);
    __syncthreads();
    for (int e = threadIdx.x; e < nv * N; e += NT) {
        const int r = e / N;
        const C z = buf[(r >> 1) * LD + (e - r * N)];
        dst[e] = ((r & 1) ? z.y : z.x) * scale;
    }
}

// ---------------------------------------------------------------- complex rows
// Per-run scalars of a lock-step batch of linear solves, in device memory:
// value k of run r at st[k * kMaxRuns + r]
constexpr int kMaxRuns = 16;
enum { RS_AR, RS_AI, RS_BR, RS_BI, RS_RR, RS_RI, RS_NORM, RS_ATOL, RS_ITERS, RS_STATUS, RS_LIVE, RS_COUNT };
__device__ __forceinline__ double run_val(const double *st, int k, int run) { return st[k * kMaxRuns + run]; }

// What the forward z pass of a lock-step batch reads: the field itself, or
// the conjugate-gradient step x += a p, p = res + b p (the new p is
// transformed on its way to memory)
template <typename T> struct CgStep {
    cpx<T> *x, *p;
    const cpx<T> *res;
    const double *st;
};

// Rows C2C forward.  STEP: the CG update above, else `in` is transformed.
template <typename T, int N, int NPEN, bool STEP>
__global__ void __launch_bounds__((NPEN *SL<T, N>::TP))
    k_rows_fwd_f(const cpx<T> *in, cpx<T> *out, long long bs, int nrows, const cpx<T> *__restrict__ twg, T scale,
                 CgStep<T> cg, const double *live) {
    if (run_off(live, blockIdx.y)) return;
    using C = cpx<T>;
    constexpr int R = SL<T, N>::first, RL = SL<T, N>::last, TP = SL<T, N>::TP, LD = N + 1;
    __shared__ C tw[N];
    __shared__ C buf[NPEN * LD];
    const int j = threadIdx.x % TP, q = threadIdx.x / TP;
    const int row = blockIdx.x * NPEN + q;
    const bool act = row < nrows;
    const long long o = (long long)blockIdx.y * bs + (long long)(act ? row : 0) * N + j;
    C v[R];
    if constexpr (STEP) {
        C r0[R], x0[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            v[r] = cg.p[o + r * TP];
            r0[r] = cg.res[o + r * TP];
            x0[r] = cg.x[o + r * TP];
        }
        const int run = blockIdx.y;
        const double ar = run_val(cg.st, RS_AR, run), ai = run_val(cg.st, RS_AI, run),
                     br = run_val(cg.st, RS_BR, run), bi = run_val(cg.st, RS_BI, run);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const C pp = v[r], xx = x0[r], rr = r0[r];
            x0[r] = C{(T)(xx.x + ar * pp.x - ai * pp.y), (T)(xx.y + ar * pp.y + ai * pp.x)};
            v[r] = C{(T)(rr.x + br * pp.x - bi * pp.y), (T)(rr.y + br * pp.y + bi * pp.x)};
        }
        if (act) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                cg.x[o + r * TP] = x0[r];
                cg.p[o + r * TP] = v[r];
            }
        }
    } else {
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] = in[o + r * TP];
    }
    for (int i = threadIdx.x; i < N; i += NPEN * TP) tw[i] = twg[i];
    dfts<T, N, RowMap<NPEN, LD>, false, false, 0, 1>(buf, tw, v, [&](auto &m, auto &u) {
        const int rl = blockIdx.x * NPEN + m.pen;
        if (!m.act || rl >= nrows) return;
        C *dst = out + (long long)blockIdx.y * bs + (long long)rl * N + m.j;
#pragma unroll
        for (int r = 0; r < RL; ++r) dst[r * (N / RL)] = C{u[r].x * scale, u[r].y * scale};
    });
}

// Inverse z pass.  MODE 0: the transform is stored.  MODE 1 to 3 finish the
// Hamiltonian product A x = x + sgn i (dt/2) (kin + v x), kin the transform:
// 1 stores A x and sums x . A x (no conjugation, two columns), 2 stores it
// and sums |A x|^2 (one column), 3 stores it.  Partial sums per run: row
// run * gridDim.x + blockIdx.x.
template <typename T> struct ApplyArgs {
    const cpx<T> *x;
    const T *v;
    double hdt;
    double *partials;
};

template <typename T, int N, int NPEN, int MODE>
__global__ void __launch_bounds__((NPEN *SL<T, N>::TP))
    k_rows_inv_f(const cpx<T> *in, cpx<T> *out, long long bs, int nrows, int ntiles, const cpx<T> *__restrict__ twg,
                 T scale, ApplyArgs<T> ap, const double *live) {
    if (run_off(live, blockIdx.y)) return;
    using C = cpx<T>;
    constexpr int R = SL<T, N>::first, RL = SL<T, N>::last, TP = SL<T, N>::TP, LD = N + 1;
    constexpr int K = MODE == 1 ? 2 : 1;
    __shared__ C tw[N];
    __shared__ C buf[NPEN * LD];
    const int j = threadIdx.x % TP, q = threadIdx.x / TP;
    for (int i = threadIdx.x; i < N; i += NPEN * TP) tw[i] = twg[i];
    double acc[K] = {};
    for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const int row = tile * NPEN + q;
        const C *src = in + (long long)blockIdx.y * bs + (long long)(row < nrows ? row : 0) * N + j;
        C v[R];
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] = src[r * TP];
        dfts<T, N, RowMap<NPEN, LD>, true, false, 0, 1>(buf, tw, v, [&](auto &m, auto &u) {
            const int rl = tile * NPEN + m.pen;
            if (!m.act || rl >= nrows) return;
            const long long o = (long long)blockIdx.y * bs + (long long)rl * N + m.j;
            if constexpr (MODE == 0) {
#pragma unroll
                for (int r = 0; r < RL; ++r) out[o + r * (N / RL)] = C{u[r].x * scale, u[r].y * scale};
            } else {
#pragma unroll
                for (int r = 0; r < RL; ++r) {
                    const C a = ap.x[o + r * (N / RL)];
                    const double vv = (double)ap.v[o + r * (N / RL)];
                    const double hr = (double)u[r].x + vv * (double)a.x, hi = (double)u[r].y + vv * (double)a.y;
                    // i * hdt * (hr + i hi) = -hdt hi + i hdt hr
                    const double orr = (double)a.x - ap.hdt * hi, oi = (double)a.y + ap.hdt * hr;
                    out[o + r * (N / RL)] = C{(T)orr, (T)oi};
                    if constexpr (MODE == 1) {
                        acc[0] += (double)a.x * orr - (double)a.y * oi;
                        acc[K - 1] += (double)a.x * oi + (double)a.y * orr;
                    } else if constexpr (MODE == 2) {
                        acc[0] += orr * orr + oi * oi;
                    }
                }
            }
        });
        if (tile + (int)gridDim.x < ntiles) __syncthreads();
    }
    if constexpr (MODE == 1 || MODE == 2) {
        block_sums<K>(acc, ap.partials + (long long)blockIdx.y * gridDim.x * K);
    }
}

// ---------------------------------------------------------------- dispatch
// Column tile: runs of 128 bytes per element row, or 256 where the workgroup
// takes that many threads
template <typename T, int N, int V> constexpr int col_tile_v() {
    int t = (V == 0 ? 128 : 256) / (2 * (int)sizeof(T));
    while (t * SL<T, N>::TP > 1024) t /= 2;
    return t;
}
// Row pairs of a workgroup: about 256 or 128 threads
template <typename T, int N, int NF, int V> constexpr int pens_v() {
    int p = (V == 0 ? 256 : 128) / (NF * SL<T, N>::TP);
    while (p > 1 && (NF * p * (N + 1) + N) * 2 * (int)sizeof(T) > 62 * 1024) --p;
    return p < 1 ? 1 : p;
}

// workgroups of a tile walk: all tiles at once up to `cap`, else equal rounds
inline int tile_blocks(long long tiles, long long cap) {
    if (tiles <= cap) return (int)tiles;
    const long long rounds = (tiles + cap - 1) / cap;
    return (int)((tiles + rounds - 1) / rounds);
}

// the odd variants have the second tile
#define OFDFT_VARIANT(var, CALL) \
    if ((var) % kTiles == 1) {        \
        CALL(1);                 \
    } else {                     \
        CALL(0);                 \
    }

template <typename T> struct SizeOps {
    void (*cols)(int var, bool inv, const cpx<T> *in, cpx<T> *out, int batch, long long bs, long long ncols,
                 long long P, long long Q, long long S, long long vp, const cpx<T> *tw, T scale, const double *live,
                 hipStream_t s, const double *gate);
    void (*xfused)(int var, cpx<T> *data, int batch, long long bs, long long ncols, long long pitch, long long vp,
                   const cpx<T> *tw, const GParams &gp, const double *live, hipStream_t s, const double *gate);
    void (*r2c)(int var, const T *in, cpx<T> *out, int batch, long long in_bs, long long out_bs, long long nrows,
                long long opitch, const cpx<T> *tw, T scale, const Prologue &pro, double *partials, int sum_slot,
                hipStream_t s, const double *gate);
    int (*r2c_tiles)(int var, int batch, long long nrows);  // its workgroups, each with a partial sum
    void (*c2r)(int var, const cpx<T> *in, T *out, int batch, long long in_bs, long long out_bs, long long nrows,
                long long ipitch, const cpx<T> *tw, T scale, hipStream_t s, const double *gate);
    void (*rows_fwd)(const cpx<T> *in, cpx<T> *out, int batch, long long bs, long long nrows, const cpx<T> *tw,
                     T scale, const CgStep<T> *cg, const double *live, hipStream_t s);
    // scale: of mode 0
    int (*rows_inv)(int mode, const cpx<T> *in, cpx<T> *out, int batch, long long bs, long long nrows,
                    const cpx<T> *tw, T scale, const ApplyArgs<T> &ap, int cap, const double *live, hipStream_t s);
};

template <typename T, int N> struct Launch {
    using C = cpx<T>;
    static constexpr int TP = SL<T, N>::TP;

    static void cols(int var, bool inv, const C *in, C *out, int batch, long long bs, long long ncols, long long P,
                     long long Q, long long S, long long vp, const C *tw, T scale, const double *live, hipStream_t s,
                     const double *gate) {
#define CALL(V)                                                                                                        \
    {                                                                                                                  \
        constexpr int TILE = col_tile_v<T, N, V>();                                                                       \
        const dim3 grid((unsigned)((ncols + TILE - 1) / TILE), (unsigned)batch);                                       \
        if (inv)                                                                                                       \
            hipLaunchKernelGGL((k_cols_f<T, N, TILE, true>), grid, dim3(TILE * TP), 0, s, in, out, bs, (unsigned)ncols, \
                               (unsigned)P, Q, S, (unsigned)vp, tw, scale, live, gate);                           \
        else                                                                                                           \
            hipLaunchKernelGGL((k_cols_f<T, N, TILE, false>), grid, dim3(TILE * TP), 0, s, in, out, bs,                 \
                               (unsigned)ncols, (unsigned)P, Q, S, (unsigned)vp, tw, scale, live, gate);          \
    }
        OFDFT_VARIANT(var, CALL)
#undef CALL
    }
    static void xfused(int var, C *data, int batch, long long bs, long long ncols, long long pitch, long long vp,
                       const C *tw, const GParams &gp, const double *live, hipStream_t s, const double *gate) {
        if constexpr (sizeof(T) == 4 && first_length(N)) {
            if (!gp.full && !gp.c2c) return xfused_ft<T>(var, data, batch, bs, ncols, pitch, vp, tw, gp, live, s, gate);
        }
        xfused_ft<double>(var, data, batch, bs, ncols, pitch, vp, tw, gp, live, s, gate);
    }
    template <typename FT>
    static void xfused_ft(int var, C *data, int batch, long long bs, long long ncols, long long pitch, long long vp,
                          const C *tw, const GParams &gp, const double *live, hipStream_t s, const double *gate) {
#define CALL(V)                                                                                                        \
    {                                                                                                                  \
        constexpr int TILE = col_tile_v<T, N, V>();                                                                       \
        const dim3 grid((unsigned)((ncols + TILE - 1) / TILE), (unsigned)batch);                                       \
        hipLaunchKernelGGL((k_xfused_f<T, FT, N, TILE>), grid, dim3(TILE * TP), 0, s, data, bs, (unsigned)ncols,           \
                           (unsigned)pitch, (unsigned)vp, tw, gp, live, gate);                                         \
    }
        OFDFT_VARIANT(var, CALL)
#undef CALL
    }
    template <int NF>
    static void r2c_nf(int var, const T *in, C *out, int nblk, long long in_bs, long long out_bs, long long nrows,
                       long long opitch, const C *tw, T scale, const Prologue &pro, double *partials, int sum_slot,
                       hipStream_t s, const double *gate) {
#define CALL(V)                                                                                                      \
    {                                                                                                                \
        constexpr int NP = pens_v<T, N, NF, V>();                                                                    \
        const long long tiles = (nrows + 2 * NP - 1) / (2 * NP);                                                     \
        const dim3 grid((unsigned)tiles, (unsigned)nblk);                                                            \
        hipLaunchKernelGGL((k_rows_r2c_f<T, N, NP, NF>), grid, dim3(NF * NP * TP), 0, s, in, out, in_bs, out_bs, nrows, \
                           (int)opitch, tw, scale, pro, partials, sum_slot, gate);                       \
    }
        OFDFT_VARIANT(var, CALL)
#undef CALL
    }
    static void r2c(int var, const T *in, C *out, int batch, long long in_bs, long long out_bs, long long nrows,
                    long long opitch, const C *tw, T scale, const Prologue &pro, double *partials, int sum_slot,
                    hipStream_t s, const double *gate) {
        if (batch == 3 && in_bs == 0)
            r2c_nf<3>(var, in, out, 1, in_bs, out_bs, nrows, opitch, tw, scale, pro, partials, sum_slot, s, gate);
        else if (batch == 2 && in_bs == 0)
            r2c_nf<2>(var, in, out, 1, in_bs, out_bs, nrows, opitch, tw, scale, pro, partials, sum_slot, s, gate);
        else
            r2c_nf<1>(var, in, out, batch, in_bs, out_bs, nrows, opitch, tw, scale, pro, partials, sum_slot, s, gate);
    }
    template <int NF> static int r2c_pens(int var) {
        return var % kTiles == 1 ? pens_v<T, N, NF, 1>() : pens_v<T, N, NF, 0>();
    }
    static int r2c_tiles(int var, int batch, long long nrows) {
        const int np = batch == 3 ? r2c_pens<3>(var) : batch == 2 ? r2c_pens<2>(var) : r2c_pens<1>(var);
        return (int)((nrows + 2 * np - 1) / (2 * np));
    }
    static void c2r(int var, const C *in, T *out, int batch, long long in_bs, long long out_bs, long long nrows,
                    long long ipitch, const C *tw, T scale, hipStream_t s, const double *gate) {
#define CALL(V)                                                                                                      \
    {                                                                                                                \
        constexpr int NP = pens_v<T, N, 1, V>();                                                                     \
        const long long tiles = (nrows + 2 * NP - 1) / (2 * NP);                                                     \
        hipLaunchKernelGGL((k_rows_c2r_f<T, N, NP>), dim3((unsigned)tiles, (unsigned)batch), dim3(NP * TP), 0, s, in, \
                           out, in_bs, out_bs, nrows, (int)ipitch, tw, scale, gate);                                 \
    }
        OFDFT_VARIANT(var, CALL)
#undef CALL
    }
    static void rows_fwd(const C *in, C *out, int batch, long long bs, long long nrows, const C *tw, T scale,
                         const CgStep<T> *cg, const double *live, hipStream_t s) {
        constexpr int NP = pens_v<T, N, 1, 0>();
        const dim3 grid((unsigned)((nrows + NP - 1) / NP), (unsigned)batch);
        if (cg)
            hipLaunchKernelGGL((k_rows_fwd_f<T, N, NP, true>), grid, dim3(NP * TP), 0, s, in, out, bs, (int)nrows, tw,
                               scale, *cg, live);
        else
            hipLaunchKernelGGL((k_rows_fwd_f<T, N, NP, false>), grid, dim3(NP * TP), 0, s, in, out, bs, (int)nrows, tw,
                               scale, CgStep<T>{}, live);
    }
    template <int MODE>
    static int inv_mode(const C *in, C *out, int batch, long long bs, long long nrows, const C *tw, T scale,
                        const ApplyArgs<T> &ap, int cap, const double *live, hipStream_t s) {
        constexpr int NP = pens_v<T, N, 1, 0>();
        const long long tiles = (nrows + NP - 1) / NP;
        const int nb = tile_blocks(tiles, cap);
        hipLaunchKernelGGL((k_rows_inv_f<T, N, NP, MODE>), dim3((unsigned)nb, (unsigned)batch), dim3(NP * TP), 0, s, in,
                           out, bs, (int)nrows, (int)tiles, tw, scale, ap, live);
        return nb;
    }
    static int rows_inv(int mode, const C *in, C *out, int batch, long long bs, long long nrows, const C *tw, T scale,
                        const ApplyArgs<T> &ap, int cap, const double *live, hipStream_t s) {
        OFDFT_REQUIRE(mode == 0 || scale == (T)1, "inverse z pass: the product takes the unscaled transform");
        if (mode == 1) return inv_mode<1>(in, out, batch, bs, nrows, tw, scale, ap, cap, live, s);
        if (mode == 2) return inv_mode<2>(in, out, batch, bs, nrows, tw, scale, ap, cap, live, s);
        if (mode == 3) return inv_mode<3>(in, out, batch, bs, nrows, tw, scale, ap, 1 << 30, live, s);
        return inv_mode<0>(in, out, batch, bs, nrows, tw, scale, ap, 1 << 30, live, s);
    }
};

template <typename T, int N> const SizeOps<T> *size_ops();

#define OFDFT_SIZE_INST(T, N)                                                                                      \
    template <> const SizeOps<T> *size_ops<T, N>() {                                                               \
        using L = Launch<T, N>;                                                                                    \
        static const SizeOps<T> ops{L::cols, L::xfused,   L::r2c,     L::r2c_tiles,                                \
                                    L::c2r,  L::rows_fwd, L::rows_inv};                                            \
        return &ops;                                                                                               \
    }

// the lengths, in groups compiled apart
#define OFDFT_SIZES_0(X, T) \
    X(T, 16) X(T, 18) X(T, 20) X(T, 22) X(T, 24) X(T, 26) X(T, 28) X(T, 30) X(T, 32) X(T, 36) X(T, 40) X(T, 42) \
    X(T, 44) X(T, 48) X(T, 50) X(T, 52) X(T, 54) X(T, 56) X(T, 60) X(T, 64)
#define OFDFT_SIZES_1(X, T) \
    X(T, 66) X(T, 70) X(T, 72) X(T, 78) X(T, 80) X(T, 84) X(T, 88) X(T, 90) X(T, 96) X(T, 98) X(T, 100) X(T, 104) \
    X(T, 108) X(T, 110) X(T, 112) X(T, 120)
#define OFDFT_SIZES_2(X, T) \
    X(T, 126) X(T, 128) X(T, 130) X(T, 132) X(T, 140) X(T, 144) X(T, 150) X(T, 154) X(T, 156) X(T, 160) X(T, 162) \
    X(T, 168) X(T, 176) X(T, 180)
#define OFDFT_SIZES_3(X, T) \
    X(T, 182) X(T, 192) X(T, 196) X(T, 198) X(T, 200) X(T, 208) X(T, 210) X(T, 216) X(T, 220) X(T, 224) X(T, 234) \
    X(T, 240) X(T, 250) X(T, 252) X(T, 256)
#define OFDFT_SIZES(X, T) OFDFT_SIZES_0(X, T) OFDFT_SIZES_1(X, T) OFDFT_SIZES_2(X, T) OFDFT_SIZES_3(X, T)

// the passes of a length, or null where it has none (fft_fixed.hip)
template <typename T> const SizeOps<T> *find_ops(int n);

}  // namespace ofdft

// Wave form of the fused physical-space pass (see physfuse.hip for the
// algorithm and the data layouts): T lanes of one wave own one theta row
// pair (j, Th-1-j) of one shell, and 64 / T row pairs share a wave.
//
// The phi transform of length n = R0 (R1) P runs as two or three Stockham
// stages whose last radix is P = n / T, so after the last inverse stage a
// lane holds the P phi points lane + T i of a field, the same points for
// every field: the pointwise products run in registers, and the forward
// transform starts from them.  The forward transform is the inverse one
// transposed (butterfly, then conjugate twiddle, the same LDS slots in the
// opposite direction), so both share their addresses and twiddle tables.
// A row pair's exchanges stay inside its wave: LDS operations of one wave
// execute in order, so no barrier separates the stages.  Only the folded
// outputs cross waves: the W (64 / T) row pairs of a workgroup are written
// as runs of consecutive theta.
//
// The zero band of the input is never loaded nor multiplied and the outputs
// beyond M are never formed (3 M <= n, the 3/2 rule).
//
// What bounds it: VALU issue and the latency of loads and LDS exchanges at two
// waves per SIMD, which the three vectors held per lane allow: without its
// loads the launch at n = 512 takes 244 us, without its stores 284 us, of 313
// us.  The workgroup form of this pass
// (physfuse.hip: a row pair per workgroup, six fields per batch, a barrier
// pair per stage) spends its time on index arithmetic, LDS bank conflicts and
// threads without a point.  FP32, per launch, workgroup -> wave form (L = M,
// N shells, Th x Ph):
//   48, 48, 72 x 144: 88 -> 41 us       86, 64, 130 x 288: 230 -> 81 us
//   170, 96, 256 x 512: 359 -> 313 us   256, 128, 384 x 768: 3422 -> 1353 us
#pragma once

#include <type_traits>

#include "fft_lds.h"
#include "lsd_internal.h"

namespace lsd {

// ------------------------------------------------ compile-time constants

constexpr double PW_PI = 3.14159265358979323846;

// cos and sin of |x| <= pi by Taylor series of the argument reduced to
// |y| <= pi/4 (error below 1e-17)
constexpr double ct_cos_small(double y) {
    double s = 1.0, t = 1.0;
    for (int k = 1; k < 12; k++) {
        t *= -y * y / ((2 * k - 1) * (2 * k));
        s += t;
    }
    return s;
}
constexpr double ct_sin_small(double y) {
    double s = y, t = y;
    for (int k = 1; k < 12; k++) {
        t *= -y * y / ((2 * k) * (2 * k + 1));
        s += t;
    }
    return s;
}
// cos(2 pi k / n), sin(2 pi k / n): octant of 8 k / n first, so that the
// multiples of an eighth turn are exact
constexpr double ct_cos(int k, int n) {
    k = ((k % n) + n) % n;
    if (2 * k > n) k = n - k;
    const bool neg = 4 * k > n;
    const int q = neg ? n - 2 * k : 2 * k;  // angle pi q / n in [0, pi/2]
    double c = 0.0;
    if (2 * q == n) c = 0.0;
    else if (4 * q > n) c = ct_sin_small(PW_PI * (n - 2 * q) / (2.0 * n));
    else c = ct_cos_small(PW_PI * q / (double)n);
    return neg ? -c : c;
}
constexpr double ct_sin(int k, int n) { return ct_cos(4 * k - n, 4 * n); }

// v exp(SG 2 pi i K / N)
template <int SG, int K, int N, typename V>
__device__ __forceinline__ V rot_ct(V v) {
    typedef decltype(V().x) S;
    constexpr int k = ((K % N) + N) % N;
    if constexpr (k == 0) return v;
    else if constexpr (4 * k == N) return cx<V>((S)-SG * v.y, (S)SG * v.x);
    else if constexpr (2 * k == N) return cx<V>(-v.x, -v.y);
    else if constexpr (4 * k == 3 * N) return cx<V>((S)SG * v.y, (S)-SG * v.x);
    else if constexpr (8 * k == N) {
        constexpr S c = (S)0.70710678118654752440;
        return cx<V>(c * (v.x - (S)SG * v.y), c * (v.y + (S)SG * v.x));
    } else if constexpr (8 * k == 3 * N) {
        constexpr S c = (S)0.70710678118654752440;
        return cx<V>(c * (-v.x - (S)SG * v.y), c * (-v.y + (S)SG * v.x));
    } else {
        constexpr S c = (S)ct_cos(k, N), s = (S)(SG * ct_sin(k, N));
        return cx<V>(v.x * c - v.y * s, v.x * s + v.y * c);
    }
}

template <int RAD, int SG, typename V>
__device__ __forceinline__ void dft_ct(V* v);

// Radix A B: A-point transforms over n1 of v[B n1 + n2], twiddles
// exp(SG 2 pi i n2 k1 / (A B)), B-point transforms over n2.
template <int A, int B, int SG, int N2, int K1, typename V>
__device__ __forceinline__ void dft_twiddle(V (&y)[B][A]) {
    if constexpr (N2 < B) {
        y[N2][K1] = rot_ct<SG, N2 * K1, A * B>(y[N2][K1]);
        dft_twiddle<A, B, SG, K1 + 1 < A ? N2 : N2 + 1, K1 + 1 < A ? K1 + 1 : 0>(y);
    }
}
template <int A, int B, int SG, typename V>
__device__ __forceinline__ void dft_ab(V* v) {
    V y[B][A];
#pragma unroll
    for (int n2 = 0; n2 < B; n2++) {
#pragma unroll
        for (int n1 = 0; n1 < A; n1++) y[n2][n1] = v[B * n1 + n2];
        dft_ct<A, SG>(y[n2]);
    }
    dft_twiddle<A, B, SG, 0, 0>(y);
#pragma unroll
    for (int k1 = 0; k1 < A; k1++) {
        V z[B];
#pragma unroll
        for (int n2 = 0; n2 < B; n2++) z[n2] = y[n2][k1];
        dft_ct<B, SG>(z);
#pragma unroll
        for (int k2 = 0; k2 < B; k2++) v[k1 + A * k2] = z[k2];
    }
}

template <int RAD, int SG, typename V>
__device__ __forceinline__ void dft_ct(V* v) {
    typedef decltype(V().x) S;
    if constexpr (RAD == 2 || RAD == 3 || RAD == 4 || RAD == 8) dft<RAD>(v, (S)SG);
    else if constexpr (RAD == 6) dft_ab<2, 3, SG>(v);
    else if constexpr (RAD == 9) dft_ab<3, 3, SG>(v);
    else if constexpr (RAD == 12) dft_ab<4, 3, SG>(v);
    else if constexpr (RAD == 16) dft_ab<4, 4, SG>(v);
    else {
        static_assert(RAD == 18, "radices 2, 3, 4, 6, 8, 9, 12, 16, 18");
        dft_ab<9, 2, SG>(v);
    }
}

// ------------------------------------------------------------------ plans

// Length N_ = R0 R1 P_ (R1 = 1: two stages).  T = N_ / P_ lanes per row
// pair; a stage of radix R has N_ / R butterflies, lane j taking j, j + T,
// ...  Between stages k and k + 1 element e sits in slot e + (e / q) p of
// the row pair's buffer, (q, p) chosen so that the lanes that LDS
// serves at once (LANES) meet distinct banks in the writes and the reads.
struct PwSwizzle {
    int q, p, cost;
};

template <int BYTES, int N_, int R0_, int R1_, int P_>
struct PwPlan {
    static constexpr int N = N_, R0 = R0_, R1 = R1_, P = P_;
    static constexpr int NS = R1 > 1 ? 3 : 2;
    static constexpr int T = N / P;
    static_assert(R0 * R1 * P == N && T <= 64, "one row pair fits a wave");
    static constexpr int G = 64 / T;  // row pairs per wave
    static constexpr int NB0 = N / R0, NB1 = N / (R1 > 1 ? R1 : N);
    static constexpr int B1 = R1 > 1 ? (NB1 + T - 1) / T : 1;
    static_assert(NB0 <= T, "the first stage takes one butterfly per lane");
    // input (and output) slots of the first (last) stage that 3 M <= N leaves
    // nonzero: i < L0 (orders 0 .. M-1) and i >= R0 - L0 (orders -(M-1) .. -1)
    static constexpr int L0 = (R0 + 2) / 3;
    static constexpr int W = G == 1 && BYTES == 8 && P <= 8 ? 8 : 4;  // waves per workgroup
    static constexpr int RP = W * G;                              // row pairs per workgroup
    // three sets of 3 P complex values stay live, 108 registers at P = 6: two
    // waves a SIMD up to P = 9, where 162 of 256 registers leave the transforms
    // too few and some spill (see the plans)
    static constexpr int WPE = BYTES == 8 && P <= 9 ? 2 : 1;

    static constexpr int LANES = 256 / BYTES;  // lanes served at once, = element slots over the 64 banks

    static constexpr int ns(int k) { return k == 0 ? 1 : k == 1 ? R0 : R0 * R1; }
    static constexpr int radix(int k) { return k == 0 ? R0 : (k == 1 && NS == 3) ? R1 : P; }
    static constexpr int wpos(int k, int j) { return (j / ns(k)) * ns(k) * radix(k) + j % ns(k); }
    static constexpr int slot(int e, int q, int p) { return e + (e / q) * p; }

    // passes LDS needs for the first write and the first read of exchange k
    static constexpr int cost(int k, int q, int p, int stride) {
        int c = 0;
        for (int rd = 0; rd < 2; rd++)
            for (int l0 = 0; l0 < 64; l0 += LANES) {
                int cnt[LANES] = {}, seen[LANES] = {}, worst = 0, ns_ = 0;
                for (int l = l0; l < l0 + LANES; l++) {
                    const int g = l / T < G ? l / T : G - 1, j = l % T;
                    const int nb = N / radix(rd ? k + 1 : k), jj = j < nb ? j : nb - 1;
                    const int s = slot(rd ? jj : wpos(k, jj), q, p) + g * stride;
                    bool dup = false;
                    for (int z = 0; z < ns_; z++) dup = dup || seen[z] == s;
                    if (dup) continue;
                    seen[ns_++] = s;
                    const int b = s % LANES;
                    cnt[b]++;
                    worst = worst > cnt[b] ? worst : cnt[b];
                }
                c += worst;
            }
        return c;
    }
    static constexpr PwSwizzle pick(int k) {
        const int nsk = ns(k + 1), nb = N / radix(k + 1);
        PwSwizzle best = {N, 0, 1 << 20};
        for (int m = 1; m <= nb / nsk; m++) {
            if ((nb / nsk) % m) continue;
            for (int p = 0; p <= 8; p++) {
                if (slot(N - 1, nsk * m, p) > N + N / 4) break;
                const int c = cost(k, nsk * m, p, 0);
                if (c < best.cost) best = PwSwizzle{nsk * m, p, c};
            }
        }
        return best;
    }
    static constexpr PwSwizzle S0 = pick(0), S1 = NS == 3 ? pick(1) : PwSwizzle{N, 0, 0};
    static constexpr int size01() {
        const int a = slot(N - 1, S0.q, S0.p) + 1, b = NS == 3 ? slot(N - 1, S1.q, S1.p) + 1 : 0;
        return a > b ? a : b;
    }
    static constexpr int pick_stride() {
        int best = size01(), bc = 1 << 20;
        for (int d = 0; d < (G > 1 ? LANES : 1); d++) {
            const int c = cost(0, S0.q, S0.p, size01() + d) + (NS == 3 ? cost(1, S1.q, S1.p, size01() + d) : 0);
            if (c < bc) {
                bc = c;
                best = size01() + d;
            }
        }
        return best;
    }
    static constexpr int BS = pick_stride();  // buffer of one row pair
    // twiddles of stage 1 (NS = 3: radix R1 over R0) and of the last stage
    static constexpr int TW1 = NS == 3 ? (R1 - 1) * R0 : 0, TWL = (P - 1) * T, TW = TW1 + TWL;
    // output staging of one row pair: orders 0 .. L0 NB0 - 1 and their negatives
    static constexpr int K = L0 * NB0;
    // row stride of the staging: the row pairs (fastest) and orders that LDS
    // serves at once in distinct banks
    static constexpr int pick_zs() {
        const int want = RP < LANES ? LANES / RP : 1;
        int z = 2 * K + 1;
        while (z % LANES != want) z++;
        return z;
    }
    static constexpr int ZS = pick_zs();
    static constexpr size_t LDS = (size_t)BYTES * (TW + RP * BS + 2 * RP * ZS);
};

template <typename R>
struct PwArgs {
    int N, Th, Th2, M, MP, gpr;  // gpr: workgroups per shell
    int nwork;
    R cor, cmag, qc, qx, scale;
    int cod, comp, mag;
    const double* gp;                  // [Th] cos(theta)
    const double* sn;                  // [Th] sin(theta)
    const typename Cx<R>::t* fourier;  // [18][N][Th][MP]
    typename Cx<R>::t* folded;         // [8][N][M][2][Th2]
    const typename Cx<R>::t* tw;       // [n] exp(2 pi i k / n)
    double* cfl;                       // CFL partial maxima [N][Th2][2] (CFL form only)
    const double* cfl_d;
    R ep, eE, ePm;
};

// Orders the LDS accesses of one wave (no instruction: a wave's LDS
// operations execute in order).
__device__ __forceinline__ void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ float2 buf_load(__amdgpu_buffer_rsrc_t r, int off, float2*) {
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    const u2 v = __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0);
    return make_float2(__uint_as_float(v.x), __uint_as_float(v.y));
}
// Keeps v in registers with an unknown value, so that what is computed from
// it (or it from) is neither moved up nor down past this point.
template <typename V>
__device__ __forceinline__ void pin(V& v) {
    asm volatile("" : "+v"(v.x), "+v"(v.y));
}

// Runs the body with the constant c, for a uniform component c = 0, 1, 2:
// registers cannot be indexed.  The comments that end the bodies keep the
// compiler from merging them again over a run-time index, which would put
// the arrays into scratch memory.
template <typename F>
__device__ __forceinline__ void by_component(int c, F&& body) {
    if (c == 0) {
        body(std::integral_constant<int, 0>{});
        asm volatile("; component 0");
    } else if (c == 1) {
        body(std::integral_constant<int, 1>{});
        asm volatile("; component 1");
    } else {
        body(std::integral_constant<int, 2>{});
        asm volatile("; component 2");
    }
}

// Physical fields in the order they are transformed: u (0-2), grad C and
// grad xi (12-17, as enabled), curl u (3-5), B (6-8), curl B (9-11).
template <typename R, class PL, bool CFL>
__global__ void __launch_bounds__(64 * PL::W) __attribute__((amdgpu_waves_per_eu(PL::WPE))) k_physwave(PwArgs<R> a) {
    typedef typename Cx<R>::t V;
    constexpr int n = PL::N, P = PL::P, T = PL::T, R0 = PL::R0, R1 = PL::R1, L0 = PL::L0, NB0 = PL::NB0;
    constexpr int NS = PL::NS, RP = PL::RP, ZS = PL::ZS, B1 = PL::B1, NT = 64 * PL::W;
    extern __shared__ unsigned char lds_raw[];
    V* twl = reinterpret_cast<V*>(lds_raw);
    V* Zo = twl + PL::TW + RP * PL::BS;  // two staging areas [RP][ZS]
    // consecutive work items of one XCD: the row-pair groups of a shell,
    // which share 128-byte lines of the folded output
    const int per = (a.nwork + 7) / 8, item = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per || item >= a.nwork) return;
    const int sh = item / a.gpr, j0 = (item - sh * a.gpr) * RP;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    // lanes past the last whole group repeat lanes of it (same values to the
    // same slots)
    const int g = min(lane / T, PL::G - 1), j = lane % T;
    const int rp = wave * PL::G + g;
    const int jp = min(j0 + rp, a.Th2 - 1), jm = a.Th - 1 - jp;
    const int N = a.N, M = a.M;
    V* X = twl + PL::TW + rp * PL::BS;

    for (int i = tid; i < PL::TW; i += NT) {
        int k;
        if (NS == 3 && i < PL::TW1) {
            const int r = i / R0 + 1, q = i % R0;
            k = q * r * (n / (R0 * R1));
        } else {
            const int i2 = i - PL::TW1, r = i2 / T + 1, q = i2 % T;
            k = q * r;
        }
        twl[i] = a.tw[k % n];
    }

    // ---- addresses: the same for every field
    const int jf = min(j, NB0 - 1);  // first-stage butterfly
    int off[2 * L0];                 // input offsets of row jp; out of range (reads 0) beyond M
    const unsigned none = 0x70000000u;
#pragma unroll
    for (int i = 0; i < 2 * L0; i++) {
        const int k = i < L0 ? jf + NB0 * i : n - jf - NB0 * (R0 - 2 * L0 + i);
        off[i] = (int)(k < M ? (unsigned)((jp * a.MP + k) * (int)sizeof(V)) : none);
    }
    const int droff = (jm - jp) * a.MP * (int)sizeof(V);  // row jm
    const size_t fsize = (size_t)N * a.Th * a.MP;         // values of one field
    V* const Xw0 = X + PL::slot(PL::wpos(0, jf), PL::S0.q, PL::S0.p);
    constexpr int RSTEP0 = PL::slot(n / PL::radix(1), PL::S0.q, PL::S0.p);  // between the reads of exchange 0
    constexpr int RSTEP1 = NS == 3 ? PL::slot(n / P, PL::S1.q, PL::S1.p) : 0;
    V* const Xrl = X + (NS == 3 ? PL::slot(j, PL::S1.q, PL::S1.p) : PL::slot(j, PL::S0.q, PL::S0.p));
    constexpr int RSTEPL = NS == 3 ? RSTEP1 : RSTEP0;
    const V* const twL = twl + PL::TW1 + j;
    int jq[B1];
#pragma unroll
    for (int q = 0; q < B1; q++) jq[q] = min(j + q * T, PL::NB1 - 1);

    V A[2 * L0], Bv[2 * L0];  // prefetched input of the next field
    auto load = [&](int f) {
        const V* base = a.fourier + (size_t)f * fsize + (size_t)sh * a.Th * a.MP;
        const auto rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<V*>(base), 0, a.Th * a.MP * (int)sizeof(V),
                                                          0x00020000);
#pragma unroll
        for (int i = 0; i < 2 * L0; i++) {
            A[i] = buf_load(rs, off[i], (V*)nullptr);
            Bv[i] = buf_load(rs, off[i] + droff, (V*)nullptr);
        }
    };
    // inverse transform of the loaded field; then loads field `next`
    auto inverse = [&](V (&v)[P], int next, bool ahead = true) {
        V z[R0];
#pragma unroll
        for (int i = 0; i < R0; i++) z[i] = cx<V>((R)0, (R)0);
#pragma unroll
        for (int i = 0; i < L0; i++) {
            V x = A[i], y = Bv[i];
            if (i == 0 && jf == 0) x.y = y.y = (R)0;  // a c2r transform drops Im of order 0
            z[i] = cx<V>(x.x - y.y, x.y + y.x);
            const V s = A[L0 + i], t = Bv[L0 + i];
            z[R0 - L0 + i] = cx<V>(s.x + t.y, t.x - s.y);
        }
        if (ahead) load(next);
        dft_ct<R0, 1>(z);
#pragma unroll
        for (int r = 0; r < R0; r++) Xw0[r] = z[r];
        wave_fence();
        if constexpr (NS == 3) {
            V y[B1][R1];
#pragma unroll
            for (int q = 0; q < B1; q++) {
                const V* s = X + PL::slot(jq[q], PL::S0.q, PL::S0.p);
#pragma unroll
                for (int r = 0; r < R1; r++) y[q][r] = s[r * RSTEP0];
                const V* t = twl + jq[q] % R0;
#pragma unroll
                for (int r = 1; r < R1; r++) y[q][r] = cmulv(y[q][r], t[(r - 1) * R0]);
                dft_ct<R1, 1>(y[q]);
            }
            wave_fence();
#pragma unroll
            for (int q = 0; q < B1; q++) {
                V* d = X + PL::slot(PL::wpos(1, jq[q]), PL::S1.q, PL::S1.p);
#pragma unroll
                for (int r = 0; r < R1; r++) d[r * R0] = y[q][r];
            }
            wave_fence();
        }
#pragma unroll
        for (int r = 0; r < P; r++) v[r] = Xrl[r * RSTEPL];
#pragma unroll
        for (int r = 1; r < P; r++) v[r] = cmulv(v[r], twL[(r - 1) * T]);
        dft_ct<P, 1>(v);
        wave_fence();
    };
    // forward transform of v (scaled by 1 / Ph first, as tra_p2s does) and
    // the fold G0 = X_j + X_mirror, G1 = X_j - X_mirror into output oid
    const size_t fstride = (size_t)N * M * 2 * a.Th2;
    int zb = 0;
    auto forward = [&](V (&v)[P], int oid) {
        const R sc = a.scale;
#pragma unroll
        for (int r = 0; r < P; r++) v[r] = cx<V>(v[r].x * sc, v[r].y * sc);
        dft_ct<P, -1>(v);
#pragma unroll
        for (int r = 0; r < P; r++) {
            if (r) {
                V w = twL[(r - 1) * T];
                w.y = -w.y;
                v[r] = cmulv(v[r], w);
            }
            Xrl[r * RSTEPL] = v[r];
        }
        wave_fence();
        if constexpr (NS == 3) {
            V y[B1][R1];
#pragma unroll
            for (int q = 0; q < B1; q++) {
                const V* s = X + PL::slot(PL::wpos(1, jq[q]), PL::S1.q, PL::S1.p);
#pragma unroll
                for (int r = 0; r < R1; r++) y[q][r] = s[r * R0];
                dft_ct<R1, -1>(y[q]);
            }
            wave_fence();
#pragma unroll
            for (int q = 0; q < B1; q++) {
                V* d = X + PL::slot(jq[q], PL::S0.q, PL::S0.p);
                const V* t = twl + jq[q] % R0;
                d[0] = y[q][0];
#pragma unroll
                for (int r = 1; r < R1; r++) {
                    V w = t[(r - 1) * R0];
                    w.y = -w.y;
                    d[r * RSTEP0] = cmulv(y[q][r], w);
                }
            }
            wave_fence();
        }
        V z[R0];
#pragma unroll
        for (int r = 0; r < R0; r++) z[r] = Xw0[r];
        wave_fence();
        dft_ct<R0, -1>(z);
        V* zo = Zo + (zb * RP + rp) * ZS;
#pragma unroll
        for (int i = 0; i < L0; i++) {
            zo[jf + NB0 * i] = z[i];                                                  // order k
            zo[PL::K + n - jf - NB0 * (R0 - L0 + i)] = z[R0 - L0 + i];  // order -k
        }
        __syncthreads();
        V* out = a.folded + oid * fstride + (size_t)sh * M * 2 * a.Th2 + j0;
#pragma unroll 1
        for (int idx = tid; idx < RP * M; idx += NT) {
            const int k = idx / RP, q = idx - k * RP;
            if (j0 + q >= a.Th2) continue;
            const V* zz = Zo + (zb * RP + q) * ZS;
            const V zk = zz[k];
            V zc = zz[k ? PL::K + k : 0];
            zc.y = -zc.y;
            const V A_ = cx<V>((R)0.5 * (zk.x + zc.x), (R)0.5 * (zk.y + zc.y));
            const V D = csubv(zk, zc);
            const V B_ = cx<V>((R)0.5 * D.y, (R)-0.5 * D.x);
            V* d = out + (size_t)k * 2 * a.Th2 + q;
            d[0] = caddv(A_, B_);
            d[a.Th2] = csubv(A_, B_);
        }
        zb ^= 1;  // the next output's staging needs no second barrier
    };

    load(LSD_P_VEL_R);
    const R sn = (R)a.sn[jp];
    const R cp = (R)a.gp[jp], cm = (R)a.gp[jm];
    __syncthreads();  // the twiddles are in place

    V u[3][P], w[3][P], nu[3][P], v[P];
    // three components (unrolled: carried through a loop, the arrays would
    // be held twice)
    auto get3 = [&](V (&d)[3][P], int f0, int after, bool ahead = true) {
        inverse(d[0], f0 + 1);
        inverse(d[1], f0 + 2);
        inverse(d[2], after, ahead);
    };
    get3(u, LSD_P_VEL_R, a.cod ? LSD_P_COD_GR : a.comp ? LSD_P_COMP_GR : LSD_P_VCURL_R);
    // advection of codensity and composition
#pragma unroll 1
    for (int s = 0; s < 2; s++) {
        if (!(s ? a.comp : a.cod)) continue;
        const int f0 = s ? LSD_P_COMP_GR : LSD_P_COD_GR;
        const int after = !s && a.comp ? LSD_P_COMP_GR : LSD_P_VCURL_R;
        const R q = s ? a.qx : a.qc;
        V sc[P];
#pragma unroll 1
        for (int c = 0; c < 3; c++) {
            inverse(v, c < 2 ? f0 + c + 1 : after);
            by_component(c, [&](auto I) {
#pragma unroll
                for (int r = 0; r < P; r++) {
                    const V t = cx<V>(-q * u[I][r].x * v[r].x, -q * u[I][r].y * v[r].y);
                    sc[r] = I ? caddv(sc[r], t) : t;
                }
            });
        }
        forward(sc, s ? NO_X : NO_C);
    }
    // advection and Coriolis
    get3(w, LSD_P_VCURL_R, LSD_P_MAG_R, a.mag);
#pragma unroll
    for (int r = 0; r < P; r++) {
        const auto one = [&](R ur, R ut, R up, R wr, R wt, R wp, R lgp, R& vr, R& vt, R& vp) {
            vr = ut * wp - up * wt;
            vt = up * wr - ur * wp;
            vp = ur * wt - ut * wr;
            vr = vr + a.cor * sn * up;
            vt = vt + a.cor * lgp * up;
            vp = vp - a.cor * (lgp * ut + sn * ur);
        };
        one(u[0][r].x, u[1][r].x, u[2][r].x, w[0][r].x, w[1][r].x, w[2][r].x, cp, nu[0][r].x, nu[1][r].x, nu[2][r].x);
        one(u[0][r].y, u[1][r].y, u[2][r].y, w[0][r].y, w[1][r].y, w[2][r].y, cm, nu[0][r].y, nu[1][r].y, nu[2][r].y);
        // formed here, not where they are used: curl u is dead from here on
        pin(nu[0][r]);
        pin(nu[1][r]);
        pin(nu[2][r]);
    }
    R cm1 = (R)-1e30, cm2 = (R)-1e30;  // CFL maxima over this lane's points (radial, horizontal)
    if (a.mag) {
        V b[3][P];
        get3(b, LSD_P_MAG_R, 0, false);
        if constexpr (CFL) {
            const R d1 = (R)a.cfl_d[2 * sh], d2 = (R)a.cfl_d[2 * sh + 1];
            const auto one = [&](R ur, R ut, R up, R br, R bt, R bp) {
                const R pr = br * br, ph = bt * bt + bp * bp;
                cm1 = fmax(cm1, pr / sqrt(pr * a.ep + d1) + fabs(ur));
                cm2 = fmax(cm2, ph / sqrt(ph * a.eE / a.ePm + d2) + sqrt(ut * ut + up * up));
            };
#pragma unroll
            for (int r = 0; r < P; r++) {
                one(u[0][r].x, u[1][r].x, u[2][r].x, b[0][r].x, b[1][r].x, b[2][r].x);
                one(u[0][r].y, u[1][r].y, u[2][r].y, b[0][r].y, b[1][r].y, b[2][r].y);
            }
        }
        // induction E = u x B
#pragma unroll 1
        for (int c = 0; c < 3; c++) {
            by_component(c, [&](auto I) {
                constexpr int I1 = (decltype(I)::value + 1) % 3;
                constexpr int I2 = (decltype(I)::value + 2) % 3;
#pragma unroll
                for (int r = 0; r < P; r++) {
                    // keeps the products of the other components from being
                    // formed ahead of their turn (3 P more live values)
                    pin(b[I1][r]);
                    pin(b[I2][r]);
                    v[r] = cx<V>(u[I1][r].x * b[I2][r].x - u[I2][r].x * b[I1][r].x,
                                 u[I1][r].y * b[I2][r].y - u[I2][r].y * b[I1][r].y);
                }
            });
            // curl B is loaded ahead during the last of the three only: three
            // vectors are live here, and held longer it would spill
            if (c == 2) load(LSD_P_MCURL_R);
            forward(v, NO_ER + c);
        }
        // Lorentz force
        get3(w, LSD_P_MCURL_R, 0, false);
#pragma unroll
        for (int r = 0; r < P; r++) {
            const R cg = a.cmag;
            nu[0][r].x = nu[0][r].x + cg * (w[1][r].x * b[2][r].x - w[2][r].x * b[1][r].x);
            nu[1][r].x = nu[1][r].x + cg * (w[2][r].x * b[0][r].x - w[0][r].x * b[2][r].x);
            nu[2][r].x = nu[2][r].x + cg * (w[0][r].x * b[1][r].x - w[1][r].x * b[0][r].x);
            nu[0][r].y = nu[0][r].y + cg * (w[1][r].y * b[2][r].y - w[2][r].y * b[1][r].y);
            nu[1][r].y = nu[1][r].y + cg * (w[2][r].y * b[0][r].y - w[0][r].y * b[2][r].y);
            nu[2][r].y = nu[2][r].y + cg * (w[0][r].y * b[1][r].y - w[1][r].y * b[0][r].y);
        }
    } else if constexpr (CFL) {
#pragma unroll
        for (int r = 0; r < P; r++) {
            cm1 = fmax(cm1, fmax(fabs(u[0][r].x), fabs(u[0][r].y)));
            cm2 = fmax(cm2, fmax(sqrt(u[1][r].x * u[1][r].x + u[2][r].x * u[2][r].x),
                                 sqrt(u[1][r].y * u[1][r].y + u[2][r].y * u[2][r].y)));
        }
    }
    if constexpr (CFL) {
        // maxima over the lanes of each row pair, through its own buffer
        X[j] = cx<V>(cm1, cm2);
        wave_fence();
        if (j == 0 && j0 + rp < a.Th2) {
#pragma unroll 1
            for (int q = 1; q < T; q++) {
                cm1 = fmax(cm1, X[q].x);
                cm2 = fmax(cm2, X[q].y);
            }
            a.cfl[((size_t)sh * a.Th2 + jp) * 2] = (double)cm1;
            a.cfl[((size_t)sh * a.Th2 + jp) * 2 + 1] = (double)cm2;
        }
        wave_fence();
    }
#pragma unroll 1
    for (int c = 0; c < 3; c++) {
        by_component(c, [&](auto I) {
#pragma unroll
            for (int r = 0; r < P; r++) v[r] = nu[I][r];
        });
        forward(v, NO_UR + c);
    }
}

// Whether a launch takes the wave form.  Its time is one row pair's chain of
// stages per round, a round being the row pairs that the registers and the LDS
// of all CUs hold, whether the round is full or not; the workgroup form's time
// is close to linear in the row pairs.  In row pairs, a round costs least +
// PW_IDLE of them and the workgroup form PW_IDLE before its first.  `least` is
// measured per plan (PW_SMALL and so on); the CFL form spills more and its
// rounds take a sixth longer.  FP32, workgroup form with 512 threads -> wave
// form: 16 shells of 64 x 128 points (512 row pairs) 30 -> 42 us, so workgroup;
// 32 shells 55 -> 44 us, so wave; at n = 512, 20 shells of 256 points 85 -> 90 us
// (the second round a quarter full), 32 shells 127 -> 105, 96 shells 353 -> 311.
// With its threads fitted to n the workgroup form stays the faster one of a
// lone run for up to twice as many row pairs, but it takes the whole GPU where
// the wave form leaves CUs to other runs: from the higher bounds twelve runs
// of 32 to 86 degrees together took 103 ms, from these 100.
constexpr long PW_IDLE = 500;
template <class PL>
bool physwave_pays(const Ctx& c, long least, bool cfl) {
    constexpr int by_regs = 4 * PL::WPE / PL::W, by_lds = (int)(163840 / PL::LDS);
    constexpr int wg = by_regs < 1 || by_lds < 1 ? 1 : by_regs < by_lds ? by_regs : by_lds;
    const long rows = (long)c.N * c.Th2, round = (long)c.ncu * wg * PL::RP;
    const long cost = least == 0 ? 0 : (cfl ? least * 6 / 5 : least) + PW_IDLE;
    return (rows + round - 1) / round * cost <= rows + PW_IDLE;
}

template <typename R, int N_, int R0_, int R1_, int P_>
int physwave_run(Ctx& c, PwArgs<R>& a, bool cfl, long least) {
    typedef PwPlan<(int)sizeof(typename Cx<R>::t), N_, R0_, R1_, P_> PL;
    if (!physwave_pays<PL>(c, least, cfl)) return 1;
    a.gpr = (c.Th2 + PL::RP - 1) / PL::RP;
    a.nwork = c.N * a.gpr;
    const dim3 g((unsigned)((a.nwork + 7) / 8 * 8));
    // algorithmic bytes: Fourier fields in, folded fields out
    const int nin = 6 + (a.mag ? 6 : 0) + (a.cod ? 3 : 0) + (a.comp ? 3 : 0);
    const int nout = 3 + (a.mag ? 3 : 0) + (a.cod ? 1 : 0) + (a.comp ? 1 : 0);
    ProfScope ps(c, LSD_K_PHYS, (double)sizeof(typename Cx<R>::t) * a.N * a.M *
                                    ((double)nin * a.Th + (double)nout * 2 * a.Th2));
    if (cfl) hipLaunchKernelGGL((k_physwave<R, PL, true>), g, dim3(64 * PL::W), PL::LDS, c.stream, a);
    else hipLaunchKernelGGL((k_physwave<R, PL, false>), g, dim3(64 * PL::W), PL::LDS, c.stream, a);
    LSD_HIP(hipGetLastError());
    return LSD_OK;
}

// The lengths each source file instantiates; 1: not one of them, or too few
// row pairs.
int physwave_f32_small(Ctx& c, PwArgs<float>& a, bool cfl);
int physwave_f32_large(Ctx& c, PwArgs<float>& a, bool cfl);
int physwave_f32_long(Ctx& c, PwArgs<float>& a, bool cfl);

#define PW_CASE(R, n, r0, r1, p, least) \
    case n: return physwave_run<R, n, r0, r1, p>(c, a, cfl, least)

// Radices: the first at most one butterfly per lane, the last (points per
// lane) 6 to 9 where the length allows, with as many of the 64 lanes in use as
// the factors give.  P = 6 holds three vectors in 256 registers; P = 8 and 9
// spill up to 368 bytes a lane (the CFL form 204 to 648).  Last, the row pairs from which
// a plan is no slower than the workgroup form with 512 threads (0: from one
// shell's on, measured from 7 shells), at L = M = n / 3 with both vector fields,
// codensity and composition.
#define PW_SMALL(R)               \
    PW_CASE(R, 36, 6, 1, 6, 180);      \
    PW_CASE(R, 48, 8, 1, 6, 220);      \
    PW_CASE(R, 54, 9, 1, 6, 250);      \
    PW_CASE(R, 64, 8, 1, 8, 500);      \
    PW_CASE(R, 72, 9, 1, 8, 320);      \
    PW_CASE(R, 96, 12, 1, 8, 430);     \
    PW_CASE(R, 108, 12, 1, 9, 500);    \
    PW_CASE(R, 128, 16, 1, 8, 850);    \
    PW_CASE(R, 144, 16, 1, 9, 650);    \
    PW_CASE(R, 162, 18, 1, 9, 600);    \
    PW_CASE(R, 192, 8, 4, 6, 420);     \
    PW_CASE(R, 216, 9, 3, 8, 500)
#define PW_LARGE(R)               \
    PW_CASE(R, 256, 8, 4, 8, 600);     \
    PW_CASE(R, 288, 8, 6, 6, 0);     \
    PW_CASE(R, 324, 9, 6, 6, 0);     \
    PW_CASE(R, 384, 8, 8, 6, 0);     \
    PW_CASE(R, 432, 9, 6, 8, 0);     \
    PW_CASE(R, 486, 9, 6, 9, 0);     \
    PW_CASE(R, 512, 8, 8, 8, 1343)

}  // namespace lsd

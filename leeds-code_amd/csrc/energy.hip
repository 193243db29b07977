// Bulk energies and their l- and m-spectra (program/io.F90:1799-1884,
// modules/variables.F90:901-957, 1267-1313): the field in qst form,
// weights w = 4 pi / (2l+1) (times 4 for m /= 0), radial integrals with
// the int r^2 dr weights.  One wave per harmonic integrates its q, s and t
// columns, then one workgroup per output (total, degree, order) sums over the
// harmonics; the order of every sum is fixed.
#include <algorithm>
#include <memory>
#include <mutex>
#include <new>

#include "lsd_internal.h"

namespace lsd {

// Sum over the lanes of a wave, in every lane.
__device__ __forceinline__ double wave_sum(double v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

// Lanes take consecutive radial points, so a column is read in whole lines
// (one work-item per column read 16 bytes of each line at a time: 99 us
// against 24 us at H = 14535, N = 96).  The stencil's neighbours come through
// the L1 cache.
constexpr int EN_WAVES = 4;
__global__ void __launch_bounds__(64 * EN_WAVES)
k_energy_h(int H, int N, int L, const int* __restrict__ hl, const int* __restrict__ hm, const double* __restrict__ r,
           const double* __restrict__ r1dr, const double* __restrict__ ll, const double* __restrict__ intr2dr,
           const double2* __restrict__ T, const double2* __restrict__ P, double* __restrict__ eh) {
    const int h = blockIdx.x * EN_WAVES + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (h >= H) return;
    const int l = hl[h];
    const double* rinv = r + 2 * N;
    const double ll1 = ll[l], rt = ll[2 * L + l];
    double w = 4.0 * 3.1415926535897931 / (double)(2 * l + 1);
    if (hm[h] != 0) w = 4.0 * w;
    const double2* Pc = P + (size_t)h * N;
    const double2* Tc = T + (size_t)h * N;
    double eq = 0.0, es = 0.0, et = 0.0;
    for (int n = lane; n < N; n += 64) {
        const double a = ll1 * rinv[n];
        const double2 pn = Pc[n], tn = Tc[n];
        const double qr = pn.x * a, qi = pn.y * a;
        // s = sqrt(l(l+1)) (1/r + d/dr) P, the 7-band stencil of r1dr
        const int lo = n - LSD_KL > 0 ? n - LSD_KL : 0;
        const int hi = n + LSD_KL < N - 1 ? n + LSD_KL : N - 1;
        double sr = 0.0, si = 0.0;
        for (int j = lo; j <= hi; j++) {
            const double b = r1dr[j * 7 + (LSD_KL + n - j)];
            const double2 pj = Pc[j];
            sr = fma(b, pj.x, sr);
            si = fma(b, pj.y, si);
        }
        sr = sr * rt;
        si = si * rt;
        const double tr = -tn.x * rt, ti = -tn.y * rt;
        eq += w * (qr * qr + qi * qi) * intr2dr[n];
        es += w * (sr * sr + si * si) * intr2dr[n];
        et += w * (tr * tr + ti * ti) * intr2dr[n];
    }
    eq = wave_sum(eq);
    es = wave_sum(es);
    et = wave_sum(et);
    if (lane == 0) {
        eh[h] = eq;
        eh[H + h] = es;
        eh[2 * H + h] = et;
    }
}

// out = [E, El[L], Em[M]], each times efac: workgroup 0 forms the total,
// 1 + l the degree-l part (its harmonics by the packed index), 1 + L + k the
// part of the k-th order (its slot is one run of harmonics).  The work-items
// take the harmonics in turn and a tree adds theirs.  (One work-item per
// output scanned all harmonics: 7.3-7.6 ms against 20 us at H = 14535.)
constexpr int ES_THREADS = 256;
__global__ void __launch_bounds__(ES_THREADS)
k_energy_sum(int H, int L, int Mp, const int* __restrict__ pidx, const Slot* __restrict__ slots,
             const int* __restrict__ mslot, double efac, const double* __restrict__ eh, double* __restrict__ out) {
    __shared__ double red[ES_THREADS / 64];
    const int t = blockIdx.x;
    double acc = 0.0;
    if (t == 0) {
        for (int i = threadIdx.x; i < 3 * H; i += ES_THREADS) acc += eh[i];
    } else if (t <= L) {
        const int l = t - 1;
        const int* row = pidx + (size_t)l * (l + 1) / 2;
        for (int m = threadIdx.x; m <= l; m += ES_THREADS) {
            const int h = row[m];
            if (h >= 0) acc += eh[h] + eh[H + h] + eh[2 * H + h];
        }
    } else {
        const Slot s = slots[mslot[t - 1 - L]];
        for (int k = threadIdx.x; k < s.len; k += ES_THREADS) {
            const int h = s.h0 + k;
            acc += eh[h] + eh[H + h] + eh[2 * H + h];
        }
    }
    acc = wave_sum(acc);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < ES_THREADS / 64; w++) acc += red[w];
        out[t] = efac * acc;
    }
}

size_t energy_scratch_doubles(const Ctx& c) { return (size_t)3 * c.H + 1 + c.L + c.M; }

int energy_run(Ctx& c, int which, double* scratch, double* E, double* El, double* Em) {
    const int H = c.H;
    double* d_eh = scratch;
    double* d_out = scratch + (size_t)3 * H;
    const double2* T = c.d_f[which ? LSD_MAG_TOR : LSD_VEL_TOR];
    const double2* P = c.d_f[which ? LSD_MAG_POL : LSD_VEL_POL];
    const double efac = which ? c.cfg.Pm / c.cfg.E : 0.5;
    hipLaunchKernelGGL(k_energy_h, dim3((H + EN_WAVES - 1) / EN_WAVES), dim3(64 * EN_WAVES), 0, c.stream, H, c.N, c.L,
                       c.d_hl, c.d_hm, c.d_r, c.d_r1dr, c.d_ll, c.d_intr2dr, T, P, d_eh);
    LSD_HIP(hipGetLastError());
    const int nt = 1 + c.L + c.M;
    hipLaunchKernelGGL(k_energy_sum, dim3(nt), dim3(ES_THREADS), 0, c.stream, H, c.L, c.Mp, c.d_pidx, c.d_slots,
                       c.d_mslot, efac, d_eh, d_out);
    LSD_HIP(hipGetLastError());
    // one copy for the total and both spectra
    const std::unique_ptr<double[]> h_out(new (std::nothrow) double[nt]);
    if (!h_out) {
        set_error("lsd_energy: out of host memory");
        return LSD_E_HIP;
    }
    LSD_HIP(hipMemcpyAsync(h_out.get(), d_out, sizeof(double) * nt, hipMemcpyDeviceToHost, c.stream));
    LSD_HIP(hipStreamSynchronize(c.stream));
    *E = h_out[0];
    if (El) std::copy(&h_out[1], &h_out[1] + c.L, El);
    if (Em) std::copy(&h_out[1] + c.L, &h_out[1] + c.L + c.M, Em);
    return LSD_OK;
}

// Scratch of lsd_energy_noalloc: the per-harmonic parts [3][H] and the
// sums [1 + L + M], one copy per GPU for the life of the process.
constexpr int ENERGY_MAX_H = 65536;
constexpr int ENERGY_MAX_LM = 2048;
constexpr size_t ENERGY_SCRATCH = (size_t)3 * ENERGY_MAX_H + 1 + ENERGY_MAX_LM;
static __device__ __align__(256) double scratch[ENERGY_SCRATCH];

constexpr int ENERGY_MAX_DEVICES = 64;
static std::mutex g_scratch_mu;
static double* g_scratch_ptr[ENERGY_MAX_DEVICES] = {};

// Device address of this device's copy of `scratch`; called once per device
// from lsd_create with that device current.
int energy_noalloc_init(int device) {
    if (device < 0 || device >= ENERGY_MAX_DEVICES) {
        set_error("lsd_create: device index beyond the static scratch table");
        return LSD_E_ARG;
    }
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (g_scratch_ptr[device]) return LSD_OK;
    double* ptr = nullptr;
    LSD_HIP(hipGetSymbolAddress((void**)&ptr, HIP_SYMBOL(scratch)));
    g_scratch_ptr[device] = ptr;
    return LSD_OK;
}

int energy_noalloc(Ctx& c, int which, double* E, double* El, double* Em) {
    if (c.H > ENERGY_MAX_H || c.L + c.M > ENERGY_MAX_LM) {
        set_error("lsd_energy_noalloc: H = " + std::to_string(c.H) + ", L + M = " + std::to_string(c.L + c.M) +
                  " exceed the static scratch (H <= 65536, L + M <= 2048); use lsd_energy");
        return LSD_E_ARG;
    }
    double* ptr = nullptr;
    {
        std::lock_guard<std::mutex> lk(g_scratch_mu);
        ptr = (c.device >= 0 && c.device < ENERGY_MAX_DEVICES) ? g_scratch_ptr[c.device] : nullptr;
    }
    if (!ptr) {
        set_error("lsd_energy_noalloc: static scratch not set up on this device");
        return LSD_E_ARG;
    }
    return energy_run(c, which, ptr, E, El, Em);
}

int energy(Ctx& c, int which, double* E, double* El, double* Em) {
    double* scratch = nullptr;
    AsyncScratch s(c.stream);
    LSD_HIP(s.alloc(&scratch, sizeof(double) * energy_scratch_doubles(c)));
    return energy_run(c, which, scratch, E, El, Em);
}

}  // namespace lsd

// pm.hip -- the PM long-range force on one GPU (one rank's whole periodic box).
//
// The reference's partmesh() with its convolution (src/partmesh.c:800-1550,
// src/conv.f90:171-229) on one rank, in FP64:
//   1. CIC deposit, mesh points at cell centres (src/partmesh.c:877-944), into the
//      periodic N^3 mesh; the scale by (N/L)^3 (:948-959) goes into the next step's factor;
//   2. hipFFT D2Z, multiply by the Green's function with sinc^-4 deconvolution and
//      the Gaussian long-range filter, pref = L^2/(pi N^3), gf(0) = pref, and pi as
//      the reference truncates it (src/conv.f90:142), hipFFT Z2D (unnormalised, as
//      2DECOMP&FFT's transforms);
//   3. one thread per particle forms the 4th-order central-difference gradient of the
//      potential and its CIC interpolation at once (the values the reference forms at
//      each particle's 8 CIC points, src/partmesh.c:1328-1550).
// acc_pm is written in the caller's order, without G (the kick applies it).
// Clustered particles pile onto few cells, so the deposit first sorts the particles
// by the lower corner of their CIC cloud: a wavefront then sums the contributions of
// each run of equal corners (segmented scan over shuffles), and the runs' sums are added
// to the mesh.  The interpolation walks the same order, so neighbouring lanes read
// neighbouring cells.  The additions' order makes the density's last bits vary.
#include <hip/hip_runtime.h>
#include <hipfft/hipfft.h>

#include <cmath>
#include <algorithm>
#include <cstring>

#include <rocprim/rocprim.hpp>

#include <stdexcept>
#include <string>

#include "../../include/photons_fmm.h"

namespace {

#define PM_CHECK(x)                                                                   \
    do {                                                                              \
        hipError_t e_ = (x);                                                          \
        if (e_ != hipSuccess) throw std::runtime_error(std::string(#x) + ": " + hipGetErrorString(e_)); \
    } while (0)
#define FFT_CHECK(x)                                                                      \
    do {                                                                                  \
        hipfftResult r_ = (x);                                                            \
        if (r_ != HIPFFT_SUCCESS) throw std::runtime_error(std::string(#x) + " failed (" + std::to_string((int)r_) + ")"); \
    } while (0)

constexpr double kPiTrunc = 3.1415926;  // src/conv.f90:142

thread_local std::string g_err;

int fail(const std::string &m)
{
    g_err = m;
    return -1;
}

struct Cic {
    int i, ii, j, jj, k, kk;
    double wi, win, wj, wjn, wk, wkn;
};

// src/partmesh.c:881-914, indices wrapped into [0, N)
__device__ __forceinline__ Cic cic(const double *p, int N, double norm, double delta)
{
    Cic c;
    int idx[3], nb[3];
    double w[3];
    for (int a = 0; a < 3; a++) {
        idx[a] = (int)(p[a] * norm);
        double wa = (p[a] - (idx[a] + 0.5) * delta) * norm;
        if (wa > 0) {
            nb[a] = idx[a] + 1;
        } else {
            wa = -wa;
            nb[a] = idx[a] - 1;
        }
        w[a] = wa;
        idx[a] = (idx[a] % N + N) % N;
        nb[a] = (nb[a] % N + N) % N;
    }
    c.i = idx[0], c.ii = nb[0], c.j = idx[1], c.jj = nb[1], c.k = idx[2], c.kk = nb[2];
    c.wi = w[0], c.wj = w[1], c.wk = w[2];
    c.win = 1.0 - w[0], c.wjn = 1.0 - w[1], c.wkn = 1.0 - w[2];
    return c;
}

__device__ __forceinline__ size_t at(int i, int j, int k, int N) { return ((size_t)i * N + j) * N + k; }

__global__ void k_fill(double *p, size_t n, double v)
{
    size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) p[t] = v;
}

// lower corner of each particle's CIC cloud (x slowest), with the particle index
__global__ void k_corner_keys(int64_t n, const double *__restrict__ pos, int N, double norm, double delta,
                              uint32_t *__restrict__ key, int32_t *__restrict__ idx)
{
    int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const Cic c = cic(pos + 3 * t, N, norm, delta);
    // the cloud covers {lo, lo+1} per axis, lo = i or the neighbour below (wrapped)
    const int lx = c.ii == (c.i + 1) % N ? c.i : c.ii;
    const int ly = c.jj == (c.j + 1) % N ? c.j : c.jj;
    const int lz = c.kk == (c.k + 1) % N ? c.k : c.kk;
    key[t] = (uint32_t)at(lx, ly, lz, N);
    idx[t] = (int32_t)t;
}

// A lane's particle t of the corner order (k: its key): its eight corner terms (as the
// reference forms them, mass * wx * wy * wz; x fastest), summed over the lanes before it in
// its run of equal corners.  tail: the run's last lane in this wavefront, with its sums.
struct RunTerms {
    double v[8];
    int cx, cy, cz;
    bool tail;
};
__device__ __forceinline__ RunTerms run_terms(int64_t t, int64_t n, uint32_t k, const double *__restrict__ pos,
                                              const int32_t *__restrict__ idx, double mass, int N, double norm,
                                              double delta)
{
    RunTerms r{};
    double (&v)[8] = r.v;
    const int lane = threadIdx.x % 64;
    const bool live = t < n;
    if (live) {
        const Cic c = cic(pos + 3 * (int64_t)idx[t], N, norm, delta);
        // weights at lo and lo + 1 per axis
        const bool ux = c.ii == (c.i + 1) % N, uy = c.jj == (c.j + 1) % N, uz = c.kk == (c.k + 1) % N;
        const double x0 = ux ? c.win : c.wi, x1 = ux ? c.wi : c.win;
        const double y0 = uy ? c.wjn : c.wj, y1 = uy ? c.wj : c.wjn;
        const double z0 = uz ? c.wkn : c.wk, z1 = uz ? c.wk : c.wkn;
        r.cx = ux ? c.i : c.ii;
        r.cy = uy ? c.j : c.jj;
        r.cz = uz ? c.k : c.kk;
        v[0] = mass * x0 * y0 * z0;
        v[1] = mass * x1 * y0 * z0;
        v[2] = mass * x0 * y1 * z0;
        v[3] = mass * x1 * y1 * z0;
        v[4] = mass * x0 * y0 * z1;
        v[5] = mass * x1 * y0 * z1;
        v[6] = mass * x0 * y1 * z1;
        v[7] = mass * x1 * y1 * z1;
    }
    // segmented inclusive scan: keys are sorted, so equal keys l-d and l mean the
    // whole stretch between them is one run
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t kd = __shfl_up(k, d, 64);
        const bool same = lane >= d && kd == k;
        if (!__ballot(same)) break;  // no run of this length: none longer
#pragma unroll
        for (int q = 0; q < 8; q++) {
            const double u = __shfl_up(v[q], d, 64);
            if (same) v[q] += u;
        }
    }
    const uint32_t knext = __shfl_down(k, 1, 64);
    r.tail = live && (lane == 63 || knext != k);
    return r;
}

// Deposit of few particles: the last lane of each run adds the run's eight sums to the
// (zeroed) mesh.
__global__ void __launch_bounds__(256) k_deposit_runs(int64_t n, const double *__restrict__ pos,
                                                      const uint32_t *__restrict__ key,
                                                      const int32_t *__restrict__ idx, double mass, int N,
                                                      double norm, double delta, double *__restrict__ mesh)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const RunTerms r = run_terms(t, n, t < n ? key[t] : 0xffffffffu, pos, idx, mass, N, norm, delta);
    if (r.tail) {
        const int x1 = (r.cx + 1) % N, y1 = (r.cy + 1) % N, z1 = (r.cz + 1) % N;
        atomicAdd(&mesh[at(r.cx, r.cy, r.cz, N)], r.v[0]);
        atomicAdd(&mesh[at(x1, r.cy, r.cz, N)], r.v[1]);
        atomicAdd(&mesh[at(r.cx, y1, r.cz, N)], r.v[2]);
        atomicAdd(&mesh[at(x1, y1, r.cz, N)], r.v[3]);
        atomicAdd(&mesh[at(r.cx, r.cy, z1, N)], r.v[4]);
        atomicAdd(&mesh[at(x1, r.cy, z1, N)], r.v[5]);
        atomicAdd(&mesh[at(r.cx, y1, z1, N)], r.v[6]);
        atomicAdd(&mesh[at(x1, y1, z1, N)], r.v[7]);
    }
}

// Deposit of many particles, without atomics on the mesh: the runs' sums are written down
// (k_run_count, a scan, k_runs), and each row of mesh points along z gathers the ones of
// the four rows of corners around it in LDS (k_deposit_rows).  The atomics of the other way
// (12M of them for 2M particles on 256^3 points) are bound by the memory side, where the
// eight XCDs' L2s meet: zeroing and deposit take 321 us there, this way 108, and the whole
// force of 2M particles 1105 -> 919 us, 16.7M 2875 -> 2484, 2M on 64^3 343 -> 306; 100,003
// on 128^3 200 -> 185 (on 64^3 114 -> 112), 30,000 on 32^3 70 -> 76 (five launches for two).
constexpr int64_t kRowsParticles = 100000;

// runs that end in each wavefront
__global__ void __launch_bounds__(256) k_run_count(int64_t n, const uint32_t *__restrict__ key, int *__restrict__ count)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int lane = threadIdx.x % 64;
    const uint64_t tails = __ballot(t < n && (lane == 63 || t + 1 == n || key[t + 1] != key[t]));
    if (lane == 0 && t < n) count[t / 64] = __popcll(tails);
}

// The runs in order: rows of corners begin at row[x N + y] (row[N N]: their number)
__global__ void __launch_bounds__(256) k_runs(int64_t n, const double *__restrict__ pos, const uint32_t *__restrict__ key,
                                              const int32_t *__restrict__ idx, double mass, int N, double norm,
                                              double delta, const int *__restrict__ off, uint32_t *__restrict__ rkey,
                                              double2 *__restrict__ sums, int64_t cap)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const RunTerms r = run_terms(t, n, t < n ? key[t] : 0xffffffffu, pos, idx, mass, N, norm, delta);
    const uint64_t tails = __ballot(r.tail);
    if (!r.tail) return;
    const int64_t at = off[t / 64] + __popcll(tails & ((1ull << (threadIdx.x % 64)) - 1ull));
    if (at >= cap) return;
    rkey[at] = key[t];
#pragma unroll
    for (int q = 0; q < 4; q++) sums[q * cap + at] = double2{r.v[q], r.v[q + 4]};  // z0, z1
}

// Run i begins the rows after run i - 1's up to its own.  More than a few of them (particles
// in few places of a large mesh) are written by the whole wavefront: with one lane's stores the
// force of 100,003 particles in a ball of 1% of the box took 449, 1621 and 8657 us on 128^3,
// 256^3 and 512^3 points, this way 184, 614 and 4565.
__global__ void __launch_bounds__(256) k_run_rows(int nwave, const int *__restrict__ off, const int *__restrict__ count,
                                                  const uint32_t *__restrict__ rkey, int N, int *__restrict__ row)
{
    const int nrun = off[nwave - 1] + count[nwave - 1];
    const int i = blockIdx.x * blockDim.x + threadIdx.x, lane = threadIdx.x % 64;
    int lo = 0, hi = -1;  // none
    if (i <= nrun) {
        lo = i ? (int)(rkey[i - 1] / (uint32_t)N) + 1 : 0;
        hi = i < nrun ? (int)(rkey[i] / (uint32_t)N) : N * N;
    }
    constexpr int kFew = 4;
    const bool many = hi - lo >= kFew;
    for (uint64_t m = __ballot(many); m; m &= m - 1) {
        const int l = __builtin_ctzll(m), e = __builtin_amdgcn_readlane(hi, l), v = __builtin_amdgcn_readlane(i, l);
        for (int r = __builtin_amdgcn_readlane(lo, l) + lane; r <= e; r += 64) row[r] = v;
    }
    if (!many)
        for (int r = lo; r <= hi; r++) row[r] = i;
}

// a wavefront for each of the four rows of corners: one below in x (q & 1), in y (q & 2)
__global__ void __launch_bounds__(256) k_deposit_rows(int N, const uint32_t *__restrict__ rkey,
                                                      const double2 *__restrict__ sums, int64_t cap,
                                                      const int *__restrict__ row, double *__restrict__ mesh)
{
    extern __shared__ double line[];  // N
    const int r = blockIdx.x, x = r / N, y = r % N, q = threadIdx.x / 64;
    for (int z = threadIdx.x; z < N; z += 256) line[z] = 0.0;
    __syncthreads();
    const int cx = q & 1 ? (x ? x : N) - 1 : x, cy = q & 2 ? (y ? y : N) - 1 : y;
    const int e = row[cx * N + cy + 1];
    const uint32_t z_at = (uint32_t)(cx * N + cy) * (uint32_t)N;
    for (int i = row[cx * N + cy] + (int)threadIdx.x % 64; i < e; i += 64) {
        const int z = (int)(rkey[i] - z_at);
        const double2 s = sums[q * cap + i];
        atomicAdd(&line[z], s.x);
        atomicAdd(&line[z + 1 == N ? 0 : z + 1], s.y);
    }
    __syncthreads();
    for (int z = threadIdx.x; z < N; z += 256) mesh[(size_t)r * N + z] = line[z];
}

__device__ __forceinline__ int wave(int a, int N) { return a > N / 2 ? a - N : a; }

__device__ __forceinline__ double sinc_pm(int v, int N)
{
    if (v == 0) return 1.0;
    const double x = kPiTrunc * v / N;
    return sin(x) / x;
}

// The half spectrum of a D2Z transform of a C-order N^3 array, [N][N][N/2+1], times the
// Green's function and the deposit's scale.  The filter and the deconvolution are products
// over the axes: their factors for the wave numbers 0 .. N/2 are formed once per workgroup
// (LDS), which then takes kGreenRows rows.  At 256^3 the sines and the exponential of every
// point took 98 us beside the 55 us that the spectrum takes to be read and written, and the
// scale a pass of its own over the mesh of 40 us.
constexpr int kGreenRows = 16;

__global__ void __launch_bounds__(256) k_green(hipfftDoubleComplex *spec, int N, double ismth2, double pref,
                                               double scale)
{
    extern __shared__ double axis[];  // N/2 + 1
    const int nc = N / 2 + 1;
    for (int v = threadIdx.x; v < nc; v += blockDim.x) {
        const double f = 1.0 / sinc_pm(v, N);
        axis[v] = exp(-(double)v * v * ismth2) * (f * f) * (f * f);
    }
    __syncthreads();
    const size_t r0 = (size_t)blockIdx.x * kGreenRows, r1 = min(r0 + kGreenRows, (size_t)N * N);
    const unsigned total = (unsigned)((r1 - r0) * nc);
    for (unsigned t = threadIdx.x; t < total; t += blockDim.x) {
        const unsigned row = t / (unsigned)nc, n = t - row * (unsigned)nc;
        const int l = abs(wave((int)((r0 + row) / N), N)), m = abs(wave((int)((r0 + row) % N), N));
        const double k2 = (double)(n * n + m * m + l * l);
        const double gf = scale * (k2 == 0.0 ? pref : pref * (axis[l] * axis[m] * axis[n]) / k2);
        hipfftDoubleComplex &z = spec[r0 * nc + t];
        z.x *= gf;
        z.y *= gf;
    }
}

// The 4th-order central differences of the potential, interpolated with the CIC weights;
// particles visited in corner order (idx), results written in the caller's order.  The
// gradient along an axis, interpolated between the cloud's two planes across it, is a sum
// over six planes, so that a particle reads 56 values of the potential, most of them out of
// the lines that its neighbours read too.  Bound by the scattered positions and forces.
// With the gradients of all mesh points formed first and 24 of them read per particle:
// 2M particles on 256^3 points 458 us, this way 167; 2M on 64^3, where a point serves 8
// particles, both within 2%.
// The error of all forces against 80-bit arithmetic is that of the mesh gradients (lattice of 48^3
// on 96^3 points 5.33e-12 and 5.34e-12, 20^3 uniform particles on 64^3 1.66e-14 and 1.67e-14).
__global__ void __launch_bounds__(256) k_interpolate(int64_t n, const double *__restrict__ pos,
                                                         const int32_t *__restrict__ idx, int N, double norm,
                                                         double delta, double invx, const double *__restrict__ phi,
                                                         double *__restrict__ acc)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const int64_t p = idx[t];
    const Cic c = cic(pos + 3 * p, N, norm, delta);
    const bool ux = c.ii == (c.i + 1) % N, uy = c.jj == (c.j + 1) % N, uz = c.kk == (c.k + 1) % N;
    const int lo[3] = {ux ? c.i : c.ii, uy ? c.j : c.jj, uz ? c.k : c.kk};
    const double w[3][2] = {{ux ? c.win : c.wi, ux ? c.wi : c.win},
                            {uy ? c.wjn : c.wj, uy ? c.wj : c.wjn},
                            {uz ? c.wkn : c.wk, uz ? c.wk : c.wkn}};
    const double f1 = 4.0 / 3.0 * invx, f2 = 1.0 / 6.0 * invx;
    double g[3][6];      // the planes' weights
    size_t o[3][6];      // their offsets
    const size_t stride[3] = {(size_t)N * N, (size_t)N, 1};
#pragma unroll
    for (int a = 0; a < 3; a++) {
        const double w0 = w[a][0], w1 = w[a][1];
        g[a][0] = f2 * w0;
        g[a][1] = f2 * w1 - f1 * w0;
        g[a][2] = -f1 * w1;
        g[a][3] = f1 * w0;
        g[a][4] = f1 * w1 - f2 * w0;
        g[a][5] = -f2 * w1;
#pragma unroll
        for (int m = 0; m < 6; m++) {
            int q = lo[a] + m - 2;
            q += q < 0 ? N : 0;
            q -= q >= N ? N : 0;
            o[a][m] = q * stride[a];
        }
    }
    // the potential from one of its values on (the first one read): the weights of a gradient add
    // to zero, and products with the whole potential would lose what its differences keep
    const double phi0 = phi[o[0][0] + o[1][2] + o[2][2]];
    double ax = 0.0, ay = 0.0, az = 0.0;
    // the planes across z and y of the cloud's own columns
#pragma unroll
    for (int i = 0; i < 6; i++)
#pragma unroll
        for (int j = 0; j < 6; j++) {
            const bool in_x = i == 2 || i == 3, in_y = j == 2 || j == 3;
            if (!in_x && !in_y) continue;
            const double *row = phi + o[0][i] + o[1][j];
            const double z0 = row[o[2][2]] - phi0, z1 = row[o[2][3]] - phi0;
            const double s = w[2][0] * z0 + w[2][1] * z1;
            if (in_y) ax += g[0][i] * w[1][j - 2] * s;
            if (in_x) ay += w[0][i - 2] * g[1][j] * s;
            if (in_x && in_y) {
                const double d = g[2][0] * (row[o[2][0]] - phi0) + g[2][1] * (row[o[2][1]] - phi0) + g[2][2] * z0 +
                                 g[2][3] * z1 + g[2][4] * (row[o[2][4]] - phi0) + g[2][5] * (row[o[2][5]] - phi0);
                az += w[0][i - 2] * w[1][j - 2] * d;
            }
        }
    acc[3 * p] = ax;
    acc[3 * p + 1] = ay;
    acc[3 * p + 2] = az;
}

inline int blocks(size_t n, int b) { return (int)((n + b - 1) / b); }

}  // namespace

struct photons_pm {
    int N = 0, device = 0;
    double L = 0, rs = 0, mass = 0;
    hipStream_t stream = nullptr;
    bool own_stream = false;
    hipfftHandle fwd = 0, inv = 0;
    double *mesh = nullptr, *io_pos = nullptr, *io_acc = nullptr;
    hipfftDoubleComplex *spec = nullptr;
    int64_t io_cap = 0;
    // corner sort: keys and particle indices (two halves each), rocPRIM temporary
    uint32_t *key = nullptr;
    int32_t *idx = nullptr;
    void *sort_tmp = nullptr;
    size_t sort_tmp_bytes = 0;
    int64_t sort_cap = 0;
    // runs of equal corners (the deposit of many particles)
    void *runs = nullptr;
    size_t runs_bytes = 0;
};

extern "C" {

const char *photons_pm_last_error(void) { return g_err.c_str(); }

int photons_pm_create(photons_pm **out, int nside, double boxsize, double rs, double mass, int device, void *stream)
{
    photons_pm *p = nullptr;
    try {
        if (!out) return fail("null handle");
        // the CIC corner keys (k_corner_keys) are 32-bit mesh indices: N^3 < 2^32
        if (nside < 8 || nside > 1624 || nside % 2)
            return fail("nside must be even, in [8, 1624] (32-bit mesh indices)");
        if (!(boxsize > 0.0) || !(rs > 0.0)) return fail("boxsize and rs must be positive");
        int ndev = 0;
        if (hipGetDeviceCount(&ndev) != hipSuccess || device < 0 || device >= ndev)
            return fail("no usable GPU for this context");
        PM_CHECK(hipSetDevice(device));
        p = new photons_pm();
        p->N = nside;
        p->L = boxsize;
        p->rs = rs;
        p->mass = mass;
        p->device = device;
        if (stream) {
            p->stream = reinterpret_cast<hipStream_t>(stream);
        } else {
            PM_CHECK(hipStreamCreateWithFlags(&p->stream, hipStreamNonBlocking));
            p->own_stream = true;
        }
        const size_t n3 = (size_t)nside * nside * nside, nc = (size_t)nside * nside * (nside / 2 + 1);
        PM_CHECK(hipMalloc(&p->mesh, sizeof(double) * n3));
        PM_CHECK(hipMalloc(&p->spec, sizeof(hipfftDoubleComplex) * nc));
        FFT_CHECK(hipfftPlan3d(&p->fwd, nside, nside, nside, HIPFFT_D2Z));
        FFT_CHECK(hipfftPlan3d(&p->inv, nside, nside, nside, HIPFFT_Z2D));
        FFT_CHECK(hipfftSetStream(p->fwd, p->stream));
        FFT_CHECK(hipfftSetStream(p->inv, p->stream));
        *out = p;
        return 0;
    } catch (const std::exception &e) {
        if (p) photons_pm_destroy(p);
        return fail(std::string("photons_pm_create: ") + e.what());
    }
}

int photons_pm_destroy(photons_pm *p)
{
    if (!p) return 0;
    (void)hipSetDevice(p->device);
    if (p->stream) (void)hipStreamSynchronize(p->stream);
    if (p->fwd) hipfftDestroy(p->fwd);
    if (p->inv) hipfftDestroy(p->inv);
    for (void *b : {(void *)p->mesh, (void *)p->spec, p->runs, (void *)p->io_pos, (void *)p->io_acc,
                    (void *)p->key, (void *)p->idx, p->sort_tmp})
        if (b) (void)hipFree(b);
    if (p->own_stream && p->stream) (void)hipStreamDestroy(p->stream);
    delete p;
    return 0;
}

// the box length of the next evaluations (the mesh shape stays): one context serves
// boxes of one mesh size and different lengths in turn
int photons_pm_set_boxsize(photons_pm *p, double boxsize)
{
    if (!p) return fail("null handle");
    if (!(boxsize > 0.0)) return fail("boxsize must be positive");
    p->L = boxsize;
    return 0;
}

// positions [n][3] in [0, L) on the device -> acc_pm [n][3], caller order, queued on
// the context's stream
int photons_pm_force_device(photons_pm *p, int64_t n, const double *d_pos, double *d_acc)
{
    try {
        if (n < 0) return fail("negative particle count");
        if (n > INT32_MAX) return fail("more than 2^31 particles");
        PM_CHECK(hipSetDevice(p->device));
        if (n == 0) return 0;
        const int N = p->N;
        const size_t n3 = (size_t)N * N * N;
        const double norm = N / p->L, delta = 1.0 / norm;
        hipStream_t st = p->stream;
        if (n > p->sort_cap) {
            for (void *b : {(void *)p->key, (void *)p->idx}) if (b) PM_CHECK(hipFree(b));
            p->key = nullptr;
            p->idx = nullptr;
            p->sort_cap = 0;
            PM_CHECK(hipMalloc(&p->key, sizeof(uint32_t) * 2 * (size_t)n));
            PM_CHECK(hipMalloc(&p->idx, sizeof(int32_t) * 2 * (size_t)n));
            p->sort_cap = n;
        }
        k_corner_keys<<<blocks(n, 256), 256, 0, st>>>(n, d_pos, N, norm, delta, p->key, p->idx);
        rocprim::double_buffer<uint32_t> kb(p->key, p->key + p->sort_cap);
        rocprim::double_buffer<int32_t> vb(p->idx, p->idx + p->sort_cap);
        unsigned bits = 1;
        while (bits < 32 && ((uint64_t)1 << bits) < (uint64_t)n3) bits++;
        size_t tmp_bytes = 0;
        PM_CHECK(rocprim::radix_sort_pairs(nullptr, tmp_bytes, kb, vb, (size_t)n, 0, bits, st));
        if (tmp_bytes > p->sort_tmp_bytes) {
            if (p->sort_tmp) PM_CHECK(hipFree(p->sort_tmp));
            p->sort_tmp = nullptr;
            p->sort_tmp_bytes = 0;
            PM_CHECK(hipMalloc(&p->sort_tmp, tmp_bytes));
            p->sort_tmp_bytes = tmp_bytes;
        }
        PM_CHECK(rocprim::radix_sort_pairs(p->sort_tmp, tmp_bytes, kb, vb, (size_t)n, 0, bits, st));
        const uint32_t *skey = kb.current();
        const int32_t *sidx = vb.current();
        // by rows: at most one run per mesh point, and one more per wavefront
        const int nwave = blocks(n, 64);
        const int64_t cap = std::min<int64_t>(n, (int64_t)n3 + nwave);
        bool rows = n >= kRowsParticles;
        size_t scan_bytes = 0, at_byte = 0;
        if (rows)
            PM_CHECK(rocprim::exclusive_scan(nullptr, scan_bytes, (int *)nullptr, (int *)nullptr, 0, (size_t)nwave,
                                             rocprim::plus<int>(), st));
        auto piece = [&](size_t bytes) {
            const size_t b = at_byte;
            at_byte += (bytes + 255) / 256 * 256;
            return b;
        };
        const size_t o_sums = piece(sizeof(double2) * 4 * cap), o_key = piece(sizeof(uint32_t) * cap),
                     o_count = piece(sizeof(int) * nwave), o_off = piece(sizeof(int) * nwave),
                     o_row = piece(sizeof(int) * ((size_t)N * N + 1)), o_scan = piece(scan_bytes);
        if (rows && at_byte > p->runs_bytes) {
            if (p->runs) PM_CHECK(hipFree(p->runs));
            p->runs = nullptr;
            p->runs_bytes = 0;
            if (hipMalloc(&p->runs, at_byte) == hipSuccess) {
                p->runs_bytes = at_byte;
            } else {  // (up to 68 bytes a particle: no memory left for them, by atomics then)
                (void)hipGetLastError();
                p->runs = nullptr;
                rows = false;
            }
        }
        if (!rows) {
            k_fill<<<blocks(n3, 256), 256, 0, st>>>(p->mesh, n3, 0.0);
            k_deposit_runs<<<blocks(n, 256), 256, 0, st>>>(n, d_pos, skey, sidx, p->mass, N, norm, delta, p->mesh);
        } else {
            char *w = static_cast<char *>(p->runs);
            double2 *sums = reinterpret_cast<double2 *>(w + o_sums);
            uint32_t *rkey = reinterpret_cast<uint32_t *>(w + o_key);
            int *count = reinterpret_cast<int *>(w + o_count), *off = reinterpret_cast<int *>(w + o_off),
                *row = reinterpret_cast<int *>(w + o_row);
            k_run_count<<<blocks(n, 256), 256, 0, st>>>(n, skey, count);
            PM_CHECK(rocprim::exclusive_scan(w + o_scan, scan_bytes, count, off, 0, (size_t)nwave, rocprim::plus<int>(),
                                             st));
            k_runs<<<blocks(n, 256), 256, 0, st>>>(n, d_pos, skey, sidx, p->mass, N, norm, delta, off, rkey, sums, cap);
            k_run_rows<<<blocks(cap + 1, 256), 256, 0, st>>>(nwave, off, count, rkey, N, row);
            k_deposit_rows<<<N * N, 256, sizeof(double) * N, st>>>(N, rkey, sums, cap, row, p->mesh);
        }
        FFT_CHECK(hipfftExecD2Z(p->fwd, p->mesh, p->spec));
        const double ismth2 = (2 * kPiTrunc * p->rs / p->L) * (2 * kPiTrunc * p->rs / p->L);
        const double pref = p->L * p->L / (kPiTrunc * (double)N * N * N);
        k_green<<<blocks((size_t)N * N, kGreenRows), 256, sizeof(double) * (N / 2 + 1), st>>>(p->spec, N, ismth2, pref,
                                                                                            norm * norm * norm);
        FFT_CHECK(hipfftExecZ2D(p->inv, p->spec, p->mesh));
        k_interpolate<<<blocks(n, 256), 256, 0, st>>>(n, d_pos, sidx, N, norm, delta, 0.5 * N / p->L, p->mesh, d_acc);
        PM_CHECK(hipGetLastError());
        return 0;
    } catch (const std::exception &e) {
        return fail(std::string("photons_pm_force_device: ") + e.what());
    }
}

int photons_pm_force_host(photons_pm *p, int64_t n, const double *pos, double *acc)
{
    try {
        if (n < 0) return fail("negative particle count");
        PM_CHECK(hipSetDevice(p->device));
        if (n == 0) return 0;
        if (n > p->io_cap) {
            if (p->io_pos) PM_CHECK(hipFree(p->io_pos));
            if (p->io_acc) PM_CHECK(hipFree(p->io_acc));
            p->io_pos = p->io_acc = nullptr;
            p->io_cap = 0;
            PM_CHECK(hipMalloc(&p->io_pos, sizeof(double) * 3 * (size_t)n));
            PM_CHECK(hipMalloc(&p->io_acc, sizeof(double) * 3 * (size_t)n));
            p->io_cap = n;
        }
        PM_CHECK(hipMemcpyAsync(p->io_pos, pos, sizeof(double) * 3 * (size_t)n, hipMemcpyHostToDevice, p->stream));
        int rc = photons_pm_force_device(p, n, p->io_pos, p->io_acc);
        if (rc) return rc;
        PM_CHECK(hipMemcpyAsync(acc, p->io_acc, sizeof(double) * 3 * (size_t)n, hipMemcpyDeviceToHost, p->stream));
        PM_CHECK(hipStreamSynchronize(p->stream));
        return 0;
    } catch (const std::exception &e) {
        return fail(std::string("photons_pm_force_host: ") + e.what());
    }
}

int photons_pm_sync(photons_pm *p)
{
    if (hipStreamSynchronize(p->stream) != hipSuccess) return fail("photons_pm_sync: stream error");
    return 0;
}

}  // extern "C"

// noalloc.hip -- compute_residual_vector_3d on caller-owned device arrays, with no
// device allocation (cism_compute_residual_vector_3d_noalloc in include/cism_gpu.h).
//
// The context entry point cism_compute_residual_vector_3d uploads host arrays into
// context buffers and reduces the two norms through the context's partial-sum
// buffer.  This variant takes device arrays in the reference's Fortran layouts and
// keeps its only scratch -- the per-workgroup partial sums of |r|^2 and |b|^2 -- in a
// file-scope __device__ array.  It calls no hipMalloc, hipFree or allocating library
// routine, so code under HIP graph capture or a serving loop that must not allocate
// can call it.  Every call on one GPU uses that GPU's copy of the array: calls that
// overlap on one GPU (other streams or threads) race on it.
#include "internal.h"

#include <mutex>

// at most this many workgroups; each leaves 2 partial sums (|r|^2, |b|^2)
#define NOALLOC_BLOCKS 1024
#define NOALLOC_THREADS 256
#define NOALLOC_MAX_DEVICES 64
// grids above this node count are rejected (the kernels' row and column arithmetic
// is 32-bit inside a column of the grid; 2^30 nodes is also 8 GB per vector)
#define NOALLOC_MAX_NODES (1LL << 30)

// the scratch: 2 * NOALLOC_BLOCKS partial sums (16 KiB); every call writes every
// entry it later reads, so nothing needs clearing between calls
static __device__ __align__(256) double scratch[2 * NOALLOC_BLOCKS];

// device address of `scratch` on each device, looked up once per device with that
// device current (each GPU holds its own copy of the array)
static double *g_scratch[NOALLOC_MAX_DEVICES];
static std::mutex g_scratch_mu;

static int scratch_on_device(int device, double **out) {
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch[device]) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            cism_set_error("residual_vector_3d_noalloc: hipGetSymbolAddress(scratch) failed on device %d: %s",
                           device, hipGetErrorString(e));
            return CISM_ERR_HIP;
        }
        g_scratch[device] = (double *)p;
    }
    *out = g_scratch[device];
    return CISM_OK;
}

// division of an n < 2^31 by a divisor fixed for a launch, exact: n m >> s with
// m = ceil(2^s / d), s = 31 + ceil(log2 d)
struct FastDiv {
    unsigned m;
    int s;
    explicit FastDiv(unsigned d) {
        int l = 0;
        while ((1ULL << l) < d) ++l;
        s = 31 + l;
        m = (unsigned)(((1ULL << s) + d - 1) / d);
    }
    __device__ int operator()(int n) const { return (int)(((unsigned long long)(unsigned)n * m) >> s); }
};

struct FGrid {
    int nz, sx, sy;            // levels, staggered extents (nx-1, ny-1)
    int ilo, ihi, jlo, jhi;    // owned staggered vertices, 0-based inclusive
    int nn;                    // nodes, at most 2^30
    FastDiv by_nz, by_sx;
};

// r = A x - b on owned active rows, 0 elsewhere; the 27 slots summed in indxA order as the
// reference's row product (pcg:2607-2645), so the vector equals the context entry point's bit
// for bit.  part[2 * block + {0, 1}] = the block's |r|^2 and |b|^2 over owned active rows, in a
// fixed order.
//
// Bound: one read of the four blocks, 864 of the 912 bytes a node needs, and on small grids
// the fetch of the code, which each wave runs once.  In the Fortran layout a node's 27
// coefficients of a block are 216 contiguous bytes, so lanes that walk their own rows touch 64
// lines per load and fetch every line again for most of the 27 slots.  Here a workgroup is one
// wave and takes tiles of 64 nodes, each in two steps, one per component: a step's two blocks
// (Auu, Auv, then Avu, Avv) are loaded as contiguous runs into registers while the step before
// sums, and pass through LDS (27.6 KB, five waves per CU; the stride of 27 doubles is odd, so the
// row reads are conflict-free).  The solution at a node's neighbours is loaded once for both
// components.  The two steps are one rolled loop, the divisions multiplications and, with one
// level, the 18 slots without a neighbour are not run through: 7 KB of code instead of 15.
// A tile without an owned active node is not read.
//
// A lane per node on its own row / tiles with both components written out and the solution
// loaded for each / now, us a call, three quarters of the columns active (all of them at one
// level): 19 x 19 x 1 nodes 8.6 / 10.0 / 8.7, 11 x 11 x 2 10.3 / 12.1 / 9.5, 34 x 34 x 10 17.4 / 12.4 / 9.6,
// 103 x 103 x 11 93 / 32 / 23, 503 x 453 x 11 2915 / 512 / 364; 34 x 34 x 10 with 5 % of the columns active
// 11.1 / 12.3 / 10.1.  Only a large grid without any row is slower than with a lane per node,
// whose waves are more: 503 x 453 x 11 15.6 / 26.3 / 22.8.
// W doubles per load: 2 when the four blocks are 16-byte aligned (a tile starts at a
// multiple of 13,824 bytes), else 1.
template <int W>
struct RowPair {
    static constexpr int N = (27 * 64 / W + 63) / 64;   // loads per lane and block
    double a[N][W], b[N][W];
};

// count coefficients of blocks A and B; past them a lane reads the last ones again.  The last
// of an odd count with W = 2 is left to pair_stage.
template <int W>
__device__ __forceinline__ void pair_load(RowPair<W> &R, const double *__restrict__ A, const double *__restrict__ B,
                                          int count, int lane) {
    typedef double vec __attribute__((ext_vector_type(W)));
    const int last = (count - W) / W * W;
#pragma unroll
    for (int t = 0; t < RowPair<W>::N; ++t) {
        const int e = min((t * 64 + lane) * W, last);
        *reinterpret_cast<vec *>(R.a[t]) = *reinterpret_cast<const vec *>(A + e);
        *reinterpret_cast<vec *>(R.b[t]) = *reinterpret_cast<const vec *>(B + e);
    }
}

// the pair to LDS, slot-minor as in memory; a lane's row is then S[27 * lane ..]
template <int W>
__device__ __forceinline__ void pair_stage(const RowPair<W> &R, const double *__restrict__ A,
                                           const double *__restrict__ B, int count, double *__restrict__ SA,
                                           double *__restrict__ SB, int lane) {
#pragma unroll
    for (int t = 0; t < RowPair<W>::N; ++t) {
        const int e = (t * 64 + lane) * W;
        if (e + W <= count)
#pragma unroll
            for (int w = 0; w < W; ++w) {
                SA[e + w] = R.a[t][w];
                SB[e + w] = R.b[t][w];
            }
    }
    if (W == 2 && (count & 1) && lane == 0) {
        SA[count - 1] = A[count - 1];
        SB[count - 1] = B[count - 1];
    }
}

template <int W>
__global__ __launch_bounds__(64) void k_resvec_fortran(
    FGrid g, const int32_t *__restrict__ av, const double *__restrict__ Auu, const double *__restrict__ Auv,
    const double *__restrict__ Avu, const double *__restrict__ Avv, const double *__restrict__ bu,
    const double *__restrict__ bv, const double *__restrict__ xu, const double *__restrict__ xv,
    double *__restrict__ ru, double *__restrict__ rv, double *__restrict__ part) {
    __shared__ alignas(16) double SA[27 * 64], SB[27 * 64];
    const int lane = threadIdx.x;
    const int cst = g.nz, rst = g.nz * g.sx;
    const int ntiles = (g.nn + 63) / 64;
    double acc[2] = {0.0, 0.0};
    // whether this lane's node of a tile has a row, and its level
    auto row_of = [&](int tile, int &k) {
        const int q = tile * 64 + lane;
        const bool in = tile < ntiles && q < g.nn;
        const int col = in ? g.by_nz(q) : 0, j = g.by_sx(col), i = col - j * g.sx;
        k = q - col * g.nz;
        return av[col] != 0 && in && i >= g.ilo && i <= g.ihi && j >= g.jlo && j <= g.jhi;
    };
    // the next tile with a row from `tile` on; the rowless ones before it are written here, each
    // after the vertices of the tile behind it are on their way
    auto find = [&](int tile, bool &row, int &k) {
        row = row_of(tile, k);
        while (tile < ntiles && !__any(row)) {
            const int q = tile * 64 + lane;
            tile += gridDim.x;
            row = row_of(tile, k);
            if (q < g.nn) {
                ru[q] = 0.0;
                rv[q] = 0.0;
            }
        }
        return tile;
    };
    // one step a component and tile: its pair of blocks is loaded while the step before sums
    RowPair<W> R;
    double x[27][2];   // the solution at the node and its neighbours
    double b0 = 0.0, b1 = 0.0, r0 = 0.0;
    // this step's tile (none yet), component, row and level, and the next step's
    int tile = ntiles, comp = 1, kk = 0, ncomp = 0, nk = 0;
    bool act = false, nact = false;
    int next = find(blockIdx.x, nact, nk);
#pragma unroll 1
    while (tile < ntiles || next < ntiles) {
        const bool have = tile < ntiles;
        const int q = tile * 64 + lane, count = 27 * min(64, g.nn - tile * 64);
        if (have) {
            const size_t o = (size_t)27 * 64 * tile;
            if (comp == 0 && act) {
                // unconditional loads, a level inside the column for one outside
#pragma unroll
                for (int kA = -1; kA <= 1; ++kA) {
                    if (kA != 0 && g.nz == 1) continue;
                    const int qk = q + (kk + kA >= 0 && kk + kA < g.nz ? kA : 0);
#pragma unroll
                    for (int h = 0; h < 9; ++h) {
                        const int qn = qk + (h % 3 - 1) * cst + (h / 3 - 1) * rst;
                        x[9 * kA + 9 + h][0] = xu[qn];
                        x[9 * kA + 9 + h][1] = xv[qn];
                    }
                }
                b0 = bu[q];
                b1 = bv[q];
            }
            pair_stage<W>(R, (comp ? Avu : Auu) + o, (comp ? Avv : Auv) + o, count, SA, SB, lane);
        }
        if (next < ntiles) {
            const size_t o = (size_t)27 * 64 * next;
            pair_load<W>(R, (ncomp ? Avu : Auu) + o, (ncomp ? Avv : Auv) + o, 27 * min(64, g.nn - next * 64), lane);
        }
        __syncthreads();
        if (have) {
            double s = 0.0;
            if (act) {   // slots in indxA order
#pragma unroll
                for (int kA = -1; kA <= 1; ++kA) {
                    if (kA != 0 && g.nz == 1) continue;
                    const bool in = kk + kA >= 0 && kk + kA < g.nz;
                    double t = s;
#pragma unroll
                    for (int m = 9 * kA + 9; m < 9 * kA + 18; ++m)
                        t = t + SA[27 * lane + m] * x[m][0] + SB[27 * lane + m] * x[m][1];
                    s = in ? t : s;
                }
                s -= comp ? b1 : b0;
            }
            if (q < g.nn) (comp ? rv : ru)[q] = s;
            if (comp == 0) {
                r0 = s;
            } else if (act) {
                acc[0] += r0 * r0 + s * s;
                acc[1] += b0 * b0 + b1 * b1;
            }
        }
        __syncthreads();
        tile = next;
        act = nact;
        kk = nk;
        comp = ncomp;
        if (ncomp && next < ntiles) next = find(next + gridDim.x, nact, nk);
        ncomp ^= 1;
    }
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        double s = acc[c];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
        if (lane == 0) part[2 * blockIdx.x + c] = s;
    }
}

// one workgroup: the nb partial pairs in a fixed order -> norms[0] = |r|, norms[1] =
// |r| / |b| (0 when |b| = 0), the reference's L2_norm and L2_norm_relative
__global__ __launch_bounds__(NOALLOC_THREADS) void k_resvec_norms(int nb, const double *__restrict__ part,
                                                                  double *__restrict__ norms) {
    __shared__ double s[2][NOALLOC_THREADS];
    double a = 0.0, b = 0.0;
    for (int t = threadIdx.x; t < nb; t += NOALLOC_THREADS) {
        a += part[2 * t];
        b += part[2 * t + 1];
    }
    s[0][threadIdx.x] = a;
    s[1][threadIdx.x] = b;
    __syncthreads();
    if (threadIdx.x >= 64) return;
    // a tree of halves: 128 and 64 apart, then within the wave
    const int t = threadIdx.x;
    double v[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        v[c] = (s[c][t] + s[c][t + 128]) + (s[c][t + 64] + s[c][t + 192]);
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) v[c] += __shfl_down(v[c], off, 64);
    }
    if (t == 0) {
        const double L2 = sqrt(v[0]), rhs = sqrt(v[1]);
        norms[0] = L2;
        norms[1] = rhs > 0.0 ? L2 / rhs : 0.0;
    }
}

extern "C" int cism_compute_residual_vector_3d_noalloc(int nx, int ny, int nz, int periodic, int device,
                                                       void *stream, const int32_t *active_vertex,
                                                       const double *Auu, const double *Auv,
                                                       const double *Avu, const double *Avv,
                                                       const double *bu, const double *bv,
                                                       const double *uvel, const double *vvel,
                                                       double *resid_u, double *resid_v, double *norms) {
    // arguments first: nothing touches the GPU before they pass
    if (nx < 7 || ny < 7 || nz < 1 || device < 0 || device >= NOALLOC_MAX_DEVICES) {
        cism_set_error("residual_vector_3d_noalloc: invalid grid nx=%d ny=%d nz=%d or device %d", nx, ny, nz,
                       device);
        return CISM_ERR_ARG;
    }
    const long long nn = (long long)nz * (nx - 1) * (ny - 1);
    if (nn > NOALLOC_MAX_NODES) {
        cism_set_error("residual_vector_3d_noalloc: %lld nodes exceed the maximum of %lld", nn, NOALLOC_MAX_NODES);
        return CISM_ERR_ARG;
    }
    if (!active_vertex || !Auu || !Auv || !Avu || !Avv || !bu || !bv || !uvel || !vvel || !resid_u ||
        !resid_v || !norms) {
        cism_set_error("residual_vector_3d_noalloc: null array");
        return CISM_ERR_ARG;
    }
    HIP_TRY(hipSetDevice(device));
    double *part = nullptr;
    CISM_TRY(scratch_on_device(device, &part));
    FGrid g{nz, nx - 1, ny - 1, 0, 0, 0, 0, (int)nn, FastDiv((unsigned)nz), FastDiv((unsigned)(nx - 1))};
    // parallel_slap.F90:661-673 (0-based): outflow domains own the west/south boundary rows
    g.ilo = (periodic ? 3 : 2) - 1;
    g.jlo = (periodic ? 3 : 2) - 1;
    g.ihi = nx - 3;
    g.jhi = ny - 3;
    long long nb = (nn + 63) / 64;   // one wave per tile of 64 nodes
    if (nb > NOALLOC_BLOCKS) nb = NOALLOC_BLOCKS;
    hipStream_t s = (hipStream_t)stream;
    // 16-byte loads of the blocks only when the caller's arrays allow them
    const bool wide = (((uintptr_t)Auu | (uintptr_t)Auv | (uintptr_t)Avu | (uintptr_t)Avv) & 15) == 0;
    hipLaunchKernelGGL(wide ? k_resvec_fortran<2> : k_resvec_fortran<1>, dim3((unsigned)nb), dim3(64), 0, s, g,
                       active_vertex, Auu, Auv, Avu, Avv, bu, bv, uvel, vvel, resid_u, resid_v, part);
    hipLaunchKernelGGL(k_resvec_norms, dim3(1), dim3(NOALLOC_THREADS), 0, s, (int)nb, part, norms);
    HIP_TRY(hipGetLastError());
    return CISM_OK;
}

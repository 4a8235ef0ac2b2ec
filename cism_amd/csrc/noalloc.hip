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

struct FGrid {
    int nz, sx, sy;            // levels, staggered extents (nx-1, ny-1)
    int ilo, ihi, jlo, jhi;    // owned staggered vertices, 0-based inclusive
    long long nn;
};

// r = A x - b on owned active rows, 0 elsewhere; the 27 slots summed in indxA order as the
// reference's row product (pcg:2607-2645), so the vector equals the context entry point's bit
// for bit.  part[2 * block + {0, 1}] = the block's |r|^2 and |b|^2 over owned active rows, in a
// fixed order.
//
// Bound: one read of the four blocks, 864 of the 912 bytes a node needs.  In the Fortran layout
// a node's 27 coefficients of a block are 216 contiguous bytes, so lanes that walk their own
// rows touch 64 lines per load and fetch every line again for most of the 27 slots (2.9 ms,
// 0.78 TB/s, at 503 x 453 x 11).  Here a workgroup is one wave and takes tiles of 64 nodes: it
// loads the tile's two blocks of one row (Auu, Auv, then Avu, Avv) as contiguous runs into
// registers, passes them through LDS (27.6 KB, four or five waves per CU; the stride of 27
// doubles is odd, so the row reads are conflict-free) and loads the next pair while it sums
// this one: 110 KB per CU in flight.  0.50 ms at that size with three quarters of the columns
// active (21.7 -> 13.5 us a call at 34 x 34 x 10).  A tile without an owned active node is
// not read.
// W doubles per load: 2 when the four blocks are 16-byte aligned (a tile starts at a
// multiple of 13,824 bytes), else 1.
template <int W>
struct RowPair {
    static constexpr int N = (27 * 64 / W + 63) / 64;   // loads per lane and block
    double a[N][W], b[N][W];
};

template <int W>
__device__ __forceinline__ void pair_load(RowPair<W> &R, const double *__restrict__ A, const double *__restrict__ B,
                                          long long q0, int count, int lane) {
    typedef double vec __attribute__((ext_vector_type(W)));
    const double *pa = A + 27 * q0, *pb = B + 27 * q0;
#pragma unroll
    for (int t = 0; t < RowPair<W>::N; ++t) {
        const int e = (t * 64 + lane) * W;
        if (e + W <= count) {
            const vec va = *reinterpret_cast<const vec *>(pa + e), vb = *reinterpret_cast<const vec *>(pb + e);
#pragma unroll
            for (int w = 0; w < W; ++w) {
                R.a[t][w] = va[w];
                R.b[t][w] = vb[w];
            }
        } else if (e < count) {   // the odd last value of the grid
            R.a[t][0] = pa[e];
            R.b[t][0] = pb[e];
        }
    }
}

template <>
__device__ __forceinline__ void pair_load<1>(RowPair<1> &R, const double *__restrict__ A,
                                             const double *__restrict__ B, long long q0, int count, int lane) {
    const double *pa = A + 27 * q0, *pb = B + 27 * q0;
#pragma unroll
    for (int t = 0; t < RowPair<1>::N; ++t) {
        const int e = t * 64 + lane;
        if (e < count) {
            R.a[t][0] = pa[e];
            R.b[t][0] = pb[e];
        }
    }
}

// the pair to LDS, slot-minor as in memory; a lane's row is then S[27 * lane ..]
template <int W>
__device__ __forceinline__ void pair_stage(const RowPair<W> &R, double *__restrict__ SA, double *__restrict__ SB,
                                           int lane) {
#pragma unroll
    for (int t = 0; t < RowPair<W>::N; ++t) {
        const int e = (t * 64 + lane) * W;
        if (e < 27 * 64)
#pragma unroll
            for (int w = 0; w < W; ++w) {
                SA[e + w] = R.a[t][w];
                SB[e + w] = R.b[t][w];
            }
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
    const long long cst = g.nz, rst = (long long)g.nz * g.sx;
    const int ntiles = (int)((g.nn + 63) / 64);
    double acc[2] = {0.0, 0.0};
    RowPair<W> R = {};
    // this lane's node of a tile: whether it has a row, and its level
    auto row_of = [&](int tile, int &k) {
        const long long q = (long long)tile * 64 + lane;
        if (q >= g.nn) return false;
        const int qi = (int)q, col = qi / g.nz;   // grids end at 2^30 nodes
        k = qi - col * g.nz;
        const int j = col / g.sx, i = col - j * g.sx;
        return i >= g.ilo && i <= g.ihi && j >= g.jlo && j <= g.jhi && av[col] != 0;
    };
    auto count_of = [&](int tile) {
        const long long left = g.nn - (long long)tile * 64;
        return (int)(left < 64 ? left : 64) * 27;
    };
    // the next tile with a row from `tile` on; the rowless ones before it are written here
    bool row = false;
    int k = 0;
    auto find = [&](int tile) {
        for (; tile < ntiles; tile += gridDim.x) {
            row = row_of(tile, k);
            if (__any(row)) break;
            const long long q = (long long)tile * 64 + lane;
            if (q < g.nn) {
                ru[q] = 0.0;
                rv[q] = 0.0;
            }
        }
        return tile;
    };
    // one component's row product from the staged pair, slots in indxA order
    auto product = [&](long long q, bool act, int kk) {
        double s = 0.0;
        if (act) {
#pragma unroll
            for (int m = 0; m < 27; ++m) {
                const int iA = m % 3 - 1, jA = (m / 3) % 3 - 1, kA = m / 9 - 1;
                if (kk + kA < 0 || kk + kA >= g.nz) continue;
                const long long qn = q + kA + iA * cst + jA * rst;
                s = s + SA[27 * lane + m] * xu[qn] + SB[27 * lane + m] * xv[qn];
            }
        }
        return s;
    };
    int tile = find(blockIdx.x);
    if (tile < ntiles) pair_load<W>(R, Auu, Auv, (long long)tile * 64, count_of(tile), lane);
    while (tile < ntiles) {
        const long long q = (long long)tile * 64 + lane;
        const bool act = row;
        const int kk = k;
        pair_stage<W>(R, SA, SB, lane);
        pair_load<W>(R, Avu, Avv, (long long)tile * 64, count_of(tile), lane);
        __syncthreads();
        const double su = product(q, act, kk);
        __syncthreads();
        pair_stage<W>(R, SA, SB, lane);
        const int next = find(tile + gridDim.x);
        if (next < ntiles) pair_load<W>(R, Auu, Auv, (long long)next * 64, count_of(next), lane);
        __syncthreads();
        const double sv = product(q, act, kk);
        __syncthreads();
        double r0 = 0.0, r1 = 0.0;
        if (act) {
            const double b0 = bu[q], b1 = bv[q];
            r0 = su - b0;
            r1 = sv - b1;
            acc[0] += r0 * r0 + r1 * r1;
            acc[1] += b0 * b0 + b1 * b1;
        }
        if (q < g.nn) {
            ru[q] = r0;
            rv[q] = r1;
        }
        tile = next;
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
    for (int w = NOALLOC_THREADS / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) {
            s[0][threadIdx.x] += s[0][threadIdx.x + w];
            s[1][threadIdx.x] += s[1][threadIdx.x + w];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const double L2 = sqrt(s[0][0]), rhs = sqrt(s[1][0]);
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
    FGrid g;
    g.nz = nz; g.sx = nx - 1; g.sy = ny - 1; g.nn = nn;
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

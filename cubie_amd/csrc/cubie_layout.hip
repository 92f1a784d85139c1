// Kernels around a launch: the layout change of per-row outputs that were
// staged run-major, and the Morton keys runs are sorted by beforehand
// (batchsolving/ordering.py).
//
// An adaptive launch writes each run's saved rows contiguously (run-major,
// element (run, row, col) at (run * rows + row) * width + col): the lanes of
// a wavefront reach their save times at different loop iterations, and a
// store into the row-major layout ((row * width + col) * n_runs + run) would
// then carry a few lanes' values into each cache line. The result layout is
// the row-major one, so the staged block is transposed afterwards: src is an
// (n_runs x inner) matrix, dst receives its (inner x n_runs) transpose, with
// inner = rows * width.
//
// The transpose goes through 64 x 64 tiles in LDS: a workgroup of 256 lanes
// reads a tile with 64-element contiguous rows from src (one 256 or 512 byte
// segment per wavefront load) and writes it back with 64-element contiguous
// rows into dst. A full tile's 16 loads per lane are issued before any of
// them is waited for, and full tiles load and store non-temporally (every
// byte is touched once). Consecutive workgroups take the tiles of an 8 x 8 group
// (run tiles x inner tiles), so the workgroups resident at one time read
// 512-element stretches of each src row and write 512-element stretches of
// each dst row. It is HBM-bound: 2 x n_runs x inner x elem_bytes per call.

#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>

#include "cubie_hip.h"
#include "cubie_order.h"

void cubie_set_last_error(const char* msg);

namespace {

constexpr int kTile = 64;
constexpr int kRowsPerPass = 4;  // 256 lanes = 64 columns x 4 rows
constexpr int kPerLane = kTile / kRowsPerPass;
constexpr int64_t kGroup = 8;    // tiles per group side
constexpr long long kMaxGrid = 1LL << 20;

template <typename T>
__global__ __launch_bounds__(256) void cubie_runs_to_rows(const T* __restrict__ src,
                                                          T* __restrict__ dst,
                                                          int64_t n_runs, int64_t inner) {
    __shared__ T tile[kTile][kTile + 1];
    const int tx = threadIdx.x & (kTile - 1);
    const int ty = threadIdx.x >> 6;
    const int64_t run_tiles = (n_runs + kTile - 1) / kTile;
    const int64_t inner_tiles = (inner + kTile - 1) / kTile;
    // groups of gr x gi tiles, inner tiles fastest inside a group
    const int64_t gr = run_tiles < kGroup ? run_tiles : kGroup;
    const int64_t gi = inner_tiles < kGroup ? inner_tiles : kGroup;
    const int64_t inner_groups = (inner_tiles + gi - 1) / gi;
    const int64_t n_slots = (run_tiles + gr - 1) / gr * inner_groups * gr * gi;
    for (int64_t t = blockIdx.x; t < n_slots; t += gridDim.x) {
        const int64_t g = t / (gr * gi);
        const int64_t l = t - g * (gr * gi);
        const int64_t tr = (g / inner_groups) * gr + l / gi;
        const int64_t ti = (g % inner_groups) * gi + l % gi;
        if (tr >= run_tiles || ti >= inner_tiles) continue;  // uniform over the workgroup
        const int64_t r0 = tr * kTile;
        const int64_t k0 = ti * kTile;
        const bool full = r0 + kTile <= n_runs && k0 + kTile <= inner;
        if (full) {
            T v[kPerLane];
            const T* s = src + (r0 + ty) * inner + k0 + tx;
#pragma unroll
            for (int p = 0; p < kPerLane; ++p) v[p] = __builtin_nontemporal_load(s + p * kRowsPerPass * inner);
#pragma unroll
            for (int p = 0; p < kPerLane; ++p) tile[ty + p * kRowsPerPass][tx] = v[p];
        } else {
            const int64_t k = k0 + tx;
            for (int i = ty; i < kTile; i += kRowsPerPass) {
                const int64_t r = r0 + i;
                if (r < n_runs && k < inner) tile[i][tx] = src[r * inner + k];
            }
        }
        __syncthreads();
        if (full) {
            T v[kPerLane];
#pragma unroll
            for (int p = 0; p < kPerLane; ++p) v[p] = tile[tx][ty + p * kRowsPerPass];
            T* d = dst + (k0 + ty) * n_runs + r0 + tx;
#pragma unroll
            for (int p = 0; p < kPerLane; ++p) __builtin_nontemporal_store(v[p], d + p * kRowsPerPass * n_runs);
        } else {
            const int64_t r = r0 + tx;
            for (int j = ty; j < kTile; j += kRowsPerPass) {
                const int64_t kk = k0 + j;
                if (r < n_runs && kk < inner) dst[kk * n_runs + r] = tile[tx][j];
            }
        }
        __syncthreads();
    }
}

struct OrderColumns {
    int n, bits;
    int index[CUBIE_ORDER_MAX_COLUMNS];
    double lo[CUBIE_ORDER_MAX_COLUMNS], span[CUBIE_ORDER_MAX_COLUMNS];
};

// One key a lane. As tensor operations this was two launches a bit and column,
// over 130 for three columns at 21 bits, 2.4 ms of launches for 131,072 runs
// with their ranges and the sort; here each column is read once. A solve of
// 131,072 sorted Hodgkin-Huxley runs went from 34.4 to 33.1 ms with it.
__global__ __launch_bounds__(256) void cubie_morton_keys(const double* __restrict__ columns,
                                                         int64_t n_runs, OrderColumns c,
                                                         long long* __restrict__ keys) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_runs) return;
    const long long levels = (1LL << c.bits) - 1;
    long long q[CUBIE_ORDER_MAX_COLUMNS];
#pragma unroll
    for (int k = 0; k < CUBIE_ORDER_MAX_COLUMNS; ++k) {
        q[k] = 0;
        if (k < c.n) {
            const double x = columns[(int64_t)c.index[k] * n_runs + i];
            const double v = rint((x - c.lo[k]) / c.span[k] * double(levels));
            q[k] = v > 0.0 ? (v < double(levels) ? (long long)v : levels) : 0;   // NaN: 0
        }
    }
    long long key = 0;
    for (int b = c.bits - 1; b >= 0; --b) {
#pragma unroll
        for (int k = 0; k < CUBIE_ORDER_MAX_COLUMNS; ++k)
            if (k < c.n) key = (key << 1) | ((q[k] >> b) & 1);
    }
    keys[i] = key;
}

}  // namespace

extern "C" {

int cubie_hip_morton_keys(const double* columns, long long n_runs, int n_cols, int bits,
                          const int* index, const double* lo, const double* span,
                          long long* keys, void* stream) {
    if (n_runs < 0 || n_cols < 1 || n_cols > CUBIE_ORDER_MAX_COLUMNS || bits < 1 || bits > 32 ||
        n_cols * bits > 63 || !index || !lo || !span) {
        cubie_set_last_error("cubie_hip_morton_keys: n_runs >= 0, 1 to 9 columns and n_cols * bits "
                             "within 63 are needed");
        return CUBIE_E_INVALID;
    }
    if (n_runs == 0) return CUBIE_OK;
    const long long blocks = (n_runs + 255) / 256;
    if (!columns || !keys || blocks > 0x7fffffffLL) {
        cubie_set_last_error("cubie_hip_morton_keys: null buffer, or too many runs");
        return CUBIE_E_INVALID;
    }
    OrderColumns c{};
    c.n = n_cols;
    c.bits = bits;
    for (int k = 0; k < n_cols; ++k) {
        if (index[k] < 0) {
            cubie_set_last_error("cubie_hip_morton_keys: negative column index");
            return CUBIE_E_INVALID;
        }
        c.index[k] = index[k];
        c.lo[k] = lo[k];
        c.span[k] = span[k];
    }
    hipLaunchKernelGGL(cubie_morton_keys, dim3(static_cast<unsigned>(blocks)), dim3(256), 0,
                       reinterpret_cast<hipStream_t>(stream), columns,
                       static_cast<int64_t>(n_runs), c, keys);
    hipError_t err = hipGetLastError();
    if (err != hipSuccess) {
        cubie_set_last_error((std::string("cubie_hip_morton_keys: ") + hipGetErrorString(err)).c_str());
        return CUBIE_E_HIP;
    }
    return CUBIE_OK;
}

int cubie_hip_runs_to_rows(const void* src, void* dst, long long n_runs, long long inner,
                           int elem_bytes, void* stream) {
    if (n_runs < 0 || inner < 0 || (elem_bytes != 4 && elem_bytes != 8)) {
        cubie_set_last_error("cubie_hip_runs_to_rows: n_runs and inner must be >= 0 and "
                             "elem_bytes 4 or 8");
        return CUBIE_E_INVALID;
    }
    if (n_runs == 0 || inner == 0) return CUBIE_OK;
    if (!src || !dst || src == dst) {
        cubie_set_last_error("cubie_hip_runs_to_rows: src and dst must be distinct device buffers");
        return CUBIE_E_INVALID;
    }
    const long long run_tiles = (n_runs + kTile - 1) / kTile;
    const long long inner_tiles = (inner + kTile - 1) / kTile;
    const long long gr = run_tiles < kGroup ? run_tiles : kGroup;
    const long long gi = inner_tiles < kGroup ? inner_tiles : kGroup;
    const long long slots = (run_tiles + gr - 1) / gr * ((inner_tiles + gi - 1) / gi) * gr * gi;
    const dim3 grid(static_cast<unsigned>(slots < kMaxGrid ? slots : kMaxGrid));
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    if (elem_bytes == 8)
        hipLaunchKernelGGL(cubie_runs_to_rows<uint64_t>, grid, dim3(256), 0, s,
                           static_cast<const uint64_t*>(src), static_cast<uint64_t*>(dst),
                           static_cast<int64_t>(n_runs), static_cast<int64_t>(inner));
    else
        hipLaunchKernelGGL(cubie_runs_to_rows<uint32_t>, grid, dim3(256), 0, s,
                           static_cast<const uint32_t*>(src), static_cast<uint32_t*>(dst),
                           static_cast<int64_t>(n_runs), static_cast<int64_t>(inner));
    hipError_t err = hipGetLastError();
    if (err != hipSuccess) {
        cubie_set_last_error((std::string("cubie_hip_runs_to_rows: ") + hipGetErrorString(err)).c_str());
        return CUBIE_E_HIP;
    }
    return CUBIE_OK;
}

}  // extern "C"

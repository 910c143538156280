// Dense neighbor matrix -> COO edge list (row-major order: atom ascending, slot ascending).
//
// Reference interface: get_neighbor_list_from_neighbor_matrix as called at
// nvalchemi/neighbors.py:92-103; the in-tree statement of its result is
// nvalchemi/models/_ops/neighbor_filter.py:255-283 (edges (E,2) rows [i, j], CSR pointer
// from the cumulative counts, shifts (E,3)).  Bound: HBM (16 B read + 20 B written per edge).
#include "common.h"
#include "scan.h"

namespace nvamd {
namespace {

constexpr int kBlock = 256;
constexpr int kLanesPerRow = 16;
constexpr int kInFlight = 3;  // entries per lane whose loads are in flight together: rows of up to 48 in one go

// A row's entries go out together (one chain of loads: the row's place, then up to 48 entries), and an entry's pair and its
// shift are one 8-byte and one 12-byte store, each group of lanes filling consecutive addresses.
// (4.3 M edges from 107 000 rows of 160 slots: 73 -> 50 us; the chain of loads bounds what is left.)
__global__ __launch_bounds__(kBlock) void coo_fill_kernel(const int32_t* __restrict__ nm,
                                                          const int32_t* __restrict__ shifts,
                                                          const int32_t* __restrict__ edge_ptr,
                                                          int n_atoms, int K, long long cap,
                                                          int32_t* __restrict__ nl,
                                                          int32_t* __restrict__ nl_shifts,
                                                          int32_t* __restrict__ counts) {
    if (counts && blockIdx.x == 0 && threadIdx.x == 0) {
        // total number of edges and whether it exceeds what the caller's buffers hold
        const int total = edge_ptr[n_atoms];
        counts[0] = total;
        counts[1] = (long long)total > cap ? 1 : 0;
    }
    const int i = (int)((blockIdx.x * (size_t)kBlock + threadIdx.x) / kLanesPerRow);
    const int sub = threadIdx.x % kLanesPerRow;
    if (i >= n_atoms) return;
    const long long e0 = edge_ptr[i];
    int cnt = edge_ptr[i + 1] - (int)e0;
    if (e0 + cnt > cap) cnt = e0 < cap ? (int)(cap - e0) : 0;
    const int32_t* row = nm + (size_t)i * K;
    const Int3* srow = shifts ? reinterpret_cast<const Int3*>(shifts) + (size_t)i * K : nullptr;
    Int2* out = reinterpret_cast<Int2*>(nl) + e0;
    Int3* sout = nl_shifts ? reinterpret_cast<Int3*>(nl_shifts) + e0 : nullptr;
    for (int k0 = sub; k0 < cnt; k0 += kInFlight * kLanesPerRow) {
        int j[kInFlight];
        Int3 s[kInFlight];
#pragma unroll
        for (int q = 0; q < kInFlight; ++q) {
            const int k = k0 + q * kLanesPerRow;
            j[q] = 0;
            s[q] = Int3{0, 0, 0};
            if (k < cnt) {
                j[q] = row[k];
                if (srow && sout) s[q] = srow[k];
            }
        }
#pragma unroll
        for (int q = 0; q < kInFlight; ++q) {
            const int k = k0 + q * kLanesPerRow;
            if (k < cnt) {
                out[k] = Int2{i, j[q]};
                if (sout) sout[k] = s[q];
            }
        }
    }
}

// The rows of a matrix behind their entries, a wave per row, in 16-byte stores.  (Padding the rows once the build has shown
// that they are wide enough, instead of filling both tensors before it, and reading what the build found at one go: 64 boxes of
// 1000 atoms with rows of 784 slots, 800 MB of padding, bound by these stores, 398 -> 350 us for list and evaluation; 512 cells
// of 8-500 atoms 418 -> 253 us; edge lists, which need no padding, of 1024 cells 383 -> 300 us.)
__global__ __launch_bounds__(kBlock) void pad_rows_kernel(const int32_t* __restrict__ nn, int n_atoms, int K, int fill,
                                                          int32_t* __restrict__ nm, int32_t* __restrict__ shifts) {
    const int i = __builtin_amdgcn_readfirstlane((int)((blockIdx.x * (size_t)kBlock + threadIdx.x) / 64));
    if (i >= n_atoms) return;
    const int n = nn[i], lane = lane_id();
    const int kept = n < 0 ? 0 : (n < K ? n : K);
    fill_words(nm + (size_t)i * K, kept, K, fill, lane);
    if (shifts) fill_words(shifts + (size_t)i * K * 3, 3 * kept, 3 * K, 0, lane);
}

// the same two numbers where there is nothing to fill
__global__ void coo_count_kernel(const int32_t* __restrict__ edge_ptr, int n_atoms, long long cap,
                                 int32_t* __restrict__ counts) {
    const int e = edge_ptr[n_atoms];
    counts[0] = e;
    counts[1] = (long long)e > cap ? 1 : 0;
}

int32_t fill(const int32_t* neighbor_matrix, const int32_t* neighbor_matrix_shifts, const int32_t* edge_ptr, int32_t n_atoms,
             int32_t max_neighbors, int64_t edge_capacity, int32_t* neighbor_list, int32_t* neighbor_list_shifts,
             int32_t* counts, hipStream_t st) {
    if (n_atoms < 0 || max_neighbors < 0 || edge_capacity < 0)
        return fail(NVAMD_ERR_INVALID_ARGUMENT, "coo: negative size");
    if (n_atoms == 0 || edge_capacity == 0 || max_neighbors == 0) {
        if (counts)
            hipLaunchKernelGGL(coo_count_kernel, dim3(1), dim3(1), 0, st, edge_ptr, n_atoms, (long long)edge_capacity, counts);
        NVAMD_LAUNCH_CHECK("coo count launch");
        return NVAMD_OK;
    }
    if (!neighbor_matrix || !edge_ptr || !neighbor_list)
        return fail(NVAMD_ERR_INVALID_ARGUMENT, "coo: null buffer");
    const size_t threads = (size_t)n_atoms * kLanesPerRow;
    hipLaunchKernelGGL(coo_fill_kernel, dim3((unsigned)((threads + kBlock - 1) / kBlock)), dim3(kBlock), 0,
                       st, neighbor_matrix, neighbor_matrix_shifts, edge_ptr, n_atoms, max_neighbors,
                       (long long)edge_capacity, neighbor_list, neighbor_list_shifts, counts);
    NVAMD_LAUNCH_CHECK("coo launch");
    return NVAMD_OK;
}

}  // namespace
}  // namespace nvamd

using namespace nvamd;

NVAMD_EXPORT int32_t nvamd_coo_workspace_bytes(int32_t n_atoms, size_t* bytes) {
    if (!bytes || n_atoms < 0) return fail(NVAMD_ERR_INVALID_ARGUMENT, "coo workspace: bad argument");
    *bytes = align_up(((size_t)scan::tiles_for((size_t)(n_atoms > 0 ? n_atoms : 1)) + 1) * sizeof(int));
    return NVAMD_OK;
}

NVAMD_EXPORT int32_t nvamd_nl_edge_ptr(const int32_t* num_neighbors, int32_t n_atoms,
                                       int32_t max_neighbors, int32_t* edge_ptr, void* workspace,
                                       size_t workspace_bytes, void* stream) {
    if (n_atoms < 0 || max_neighbors < 0) return fail(NVAMD_ERR_INVALID_ARGUMENT, "edge_ptr: negative size");
    if (!edge_ptr || (n_atoms > 0 && !num_neighbors))
        return fail(NVAMD_ERR_INVALID_ARGUMENT, "edge_ptr: null buffer");
    size_t need = 0;
    nvamd_coo_workspace_bytes(n_atoms, &need);
    if (!workspace || workspace_bytes < need)
        return fail(NVAMD_ERR_WORKSPACE_TOO_SMALL, "edge_ptr: workspace %zu < %zu bytes", workspace_bytes, need);
    if ((long long)n_atoms * max_neighbors > 0x7fffffffLL)
        return fail(NVAMD_ERR_UNSUPPORTED, "edge_ptr: N*K exceeds int32 edge offsets");
    hipStream_t st = static_cast<hipStream_t>(stream);
    scan::exclusive(scan::LoadClamped{num_neighbors, max_neighbors}, nullptr, n_atoms,
                    scan::tiles_for((size_t)n_atoms), static_cast<int*>(workspace), edge_ptr, st);
    NVAMD_LAUNCH_CHECK("edge_ptr launch");
    return NVAMD_OK;
}

NVAMD_EXPORT int32_t nvamd_nl_matrix_to_coo(const int32_t* neighbor_matrix,
                                            const int32_t* neighbor_matrix_shifts,
                                            const int32_t* edge_ptr, int32_t n_atoms,
                                            int32_t max_neighbors, int64_t edge_capacity,
                                            int32_t* neighbor_list, int32_t* neighbor_list_shifts,
                                            void* stream) {
    return fill(neighbor_matrix, neighbor_matrix_shifts, edge_ptr, n_atoms, max_neighbors, edge_capacity, neighbor_list,
                neighbor_list_shifts, nullptr, static_cast<hipStream_t>(stream));
}

NVAMD_EXPORT int32_t nvamd_nl_coo_from_matrix(const int32_t* neighbor_matrix, const int32_t* neighbor_matrix_shifts,
                                              const int32_t* num_neighbors, int32_t n_atoms, int32_t max_neighbors,
                                              int64_t edge_capacity, int32_t* edge_ptr, int32_t* neighbor_list,
                                              int32_t* neighbor_list_shifts, int32_t* counts, void* workspace,
                                              size_t workspace_bytes, void* stream) {
    if (!counts) return fail(NVAMD_ERR_INVALID_ARGUMENT, "coo: null counts");
    int32_t rc = nvamd_nl_edge_ptr(num_neighbors, n_atoms, max_neighbors, edge_ptr, workspace, workspace_bytes, stream);
    if (rc != NVAMD_OK) return rc;
    return fill(neighbor_matrix, neighbor_matrix_shifts, edge_ptr, n_atoms, max_neighbors, edge_capacity, neighbor_list,
                neighbor_list_shifts, counts, static_cast<hipStream_t>(stream));
}

NVAMD_EXPORT int32_t nvamd_nl_pad_rows(const int32_t* num_neighbors, int32_t n_atoms, int32_t max_neighbors, int32_t fill_value,
                                       int32_t* neighbor_matrix, int32_t* neighbor_matrix_shifts, void* stream) {
    if (n_atoms < 0 || max_neighbors < 0 || (long long)max_neighbors * 3 > 0x7fffffffLL)
        return fail(NVAMD_ERR_INVALID_ARGUMENT, "pad rows: bad size");
    if (n_atoms == 0 || max_neighbors == 0) return NVAMD_OK;
    if (!num_neighbors || !neighbor_matrix) return fail(NVAMD_ERR_INVALID_ARGUMENT, "pad rows: null buffer");
    const size_t threads = (size_t)n_atoms * 64;
    hipLaunchKernelGGL(pad_rows_kernel, dim3((unsigned)((threads + kBlock - 1) / kBlock)), dim3(kBlock), 0,
                       static_cast<hipStream_t>(stream), num_neighbors, n_atoms, max_neighbors, fill_value, neighbor_matrix,
                       neighbor_matrix_shifts);
    NVAMD_LAUNCH_CHECK("pad rows launch");
    return NVAMD_OK;
}

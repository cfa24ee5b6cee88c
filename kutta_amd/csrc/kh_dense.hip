// FP64 dense coarsest-level solve for the mixed-precision AMG path (no
// reference counterpart): the coarse operator, stored FP32 in CSR, is
// expanded into a dense FP64 matrix and inverted in place by blocked
// Gauss-Jordan elimination without pivoting (the operator is symmetric
// positive definite: a pinned M-matrix and its Galerkin products). Per block
// of kGjBlock pivots K:
//   P = A_KK^-1 (one workgroup, element-wise Gauss-Jordan), A_KK = P
//   A_KJ = P A_KJ                (row panel, J outside K)
//   A_IJ -= A_IK A_KJ            (trailing update, I and J outside K)
//   A_IK = -A_IK P               (column panel)
// The three products are 64 x 64 tiles on the FP64 MFMA
// (v_mfma_f64_16x16x4_f64). Each V-cycle then applies the inverse as an FP64
// matrix-vector product, one workgroup per row.
#include "kh_device_math.hpp"

namespace kh {
namespace {

typedef double f64x4 __attribute__((ext_vector_type(4)));
constexpr int kGjBlock = 64;          // pivots per block, and the tile edge
constexpr int kGjStride = kGjBlock + 2;  // LDS row stride (doubles): half a wavefront's L operands fall on all banks

__global__ void __launch_bounds__(kBlock) k_dense_clear(long count, double* __restrict__ dense) {
  const long i = long(blockIdx.x) * kBlock + threadIdx.x;
  if (i < count) dense[i] = 0.0;
}
__global__ void __launch_bounds__(kBlock) k_dense_scatter(int n, const int* __restrict__ rows,
    const int* __restrict__ cols, const float* __restrict__ values, double* __restrict__ dense) {
  const int i = int(blockIdx.x) * kBlock + int(threadIdx.x);
  if (i >= n) return;
  for (int j = rows[i]; j < rows[i + 1]; ++j) dense[long(i) * n + cols[j]] += double(values[j]);
}

// A 64 x 64 tile on one 256-thread workgroup: thread (wave w, lane l) holds
// column 16 w + l % 16 and the rows of its 16 slots, slot m being row
// 4 m + l / 16. That is the accumulator of v_mfma_f64_16x16x4_f64 (register q
// of row block br is slot 4 br + q: the FP64 accumulator interleaves rows;
// checked against a CPU product on the device), for which the lane supplies
// L[16 br + l%16][4 s + l/16] and R[4 s + l/16][16 w + l%16]: a tile's R comes
// from memory straight into that layout, L through LDS.
constexpr int kSlots = 16;
__device__ __forceinline__ int tile_row(int m) { return 4 * m + ((threadIdx.x & 63) >> 4); }
__device__ __forceinline__ int tile_col() { return 16 * int(threadIdx.x >> 6) + int(threadIdx.x & 15); }
// The tile at (i0, j0), zero from `rows` and `cols` on. All 16 loads are in
// flight before the first is used.
__device__ __forceinline__ void load_slots(double (&v)[kSlots], const double* __restrict__ a, int n, int i0, int j0,
                                           int rows, int cols) {
  const int c = tile_col();
#pragma unroll
  for (int m = 0; m < kSlots; ++m)
    v[m] = a[long(i0 + min(tile_row(m), rows - 1)) * n + j0 + min(c, cols - 1)];
#pragma unroll
  for (int m = 0; m < kSlots; ++m)
    if (tile_row(m) >= rows || c >= cols) v[m] = 0.0;
}
// The tile as the left factor: consecutive threads load consecutive columns.
__device__ __forceinline__ void load_rows(double (&v)[kSlots], const double* __restrict__ a, int n, int i0, int j0,
                                          int rows, int cols) {
  const int c = threadIdx.x & 63, r0 = threadIdx.x >> 6;
#pragma unroll
  for (int m = 0; m < kSlots; ++m)
    v[m] = a[long(i0 + min(r0 + 4 * m, rows - 1)) * n + j0 + min(c, cols - 1)];
#pragma unroll
  for (int m = 0; m < kSlots; ++m)
    if (r0 + 4 * m >= rows || c >= cols) v[m] = 0.0;
}
__device__ __forceinline__ void stage_rows(double* L, const double (&v)[kSlots]) {
  const int c = threadIdx.x & 63, r0 = threadIdx.x >> 6;
#pragma unroll
  for (int m = 0; m < kSlots; ++m) L[(r0 + 4 * m) * kGjStride + c] = v[m];
}
// L R for the staged L and this thread's R values.
__device__ __forceinline__ void tile_product(const double* L, const double (&rv)[kSlots], double (&out)[kSlots]) {
  const int lane = threadIdx.x & 63;
  const double* l = L + (lane & 15) * kGjStride + (lane >> 4);
  f64x4 acc[4] = {};
#pragma unroll
  for (int s = 0; s < kSlots; ++s) {
#pragma unroll
    for (int br = 0; br < 4; ++br)
      acc[br] = __builtin_amdgcn_mfma_f64_16x16x4f64(l[16 * br * kGjStride + 4 * s], rv[s], acc[br], 0, 0, 0);
  }
#pragma unroll
  for (int m = 0; m < kSlots; ++m) out[m] = acc[m / 4][m % 4];
}
__device__ __forceinline__ void store_slots(const double (&v)[kSlots], double* __restrict__ a, int n, int i0, int j0,
                                            int rows, int cols) {
  const int c = tile_col();
#pragma unroll
  for (int m = 0; m < kSlots; ++m)
    if (tile_row(m) < rows && c < cols) a[long(i0 + tile_row(m)) * n + j0 + c] = v[m];
}

// The inverse of the b x b tile held in slots: element-wise Gauss-Jordan,
// pivot by pivot with the pivot's reciprocal r = 1/p (a_pp' = r,
// a_pj' = a_pj r, a_ip' = -a_ip r, a_ij' = a_ij - a_ip (a_pj r)). Rows and
// columns from b on are taken as the identity's, which leaves the rest as it
// is. A pivot is one barrier: its row and column go out through LDS (two
// buffers in turn) and every thread forms r itself. The slots turn by one
// every four pivots, so that the pivot's row is always in slot 0 and no
// register is indexed at run time. 64 pivots: 80 us before (four entries of
// 1024 threads in LDS, two barriers each, and a launch of its own).
__device__ __forceinline__ void invert_slots(double (&t)[kSlots], int b, double* lds) {
  const int lane = threadIdx.x & 63, sub = lane >> 4, j = tile_col();
#pragma unroll
  for (int m = 0; m < kSlots; ++m)
    if (tile_row(m) >= b || j >= b) t[m] = tile_row(m) == j ? 1.0 : 0.0;
  for (int group = 0; group < kSlots; ++group) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int q = 4 * group + u;
      double* row = lds + (u & 1) * 2 * kGjBlock;
      double* col = row + kGjBlock;  // [sub][slot]
      if (sub == u) row[j] = t[0];
      if (j == q) {
#pragma unroll
        for (int m = 0; m < kSlots; ++m) col[sub * kSlots + m] = t[m];
      }
      __syncthreads();
      const double r = 1.0 / row[q], scaled = row[j] * r;
      const bool mine = j == q;
      double c[kSlots];
#pragma unroll
      for (int m = 0; m < kSlots; ++m) c[m] = col[sub * kSlots + m];
#pragma unroll
      for (int m = 0; m < kSlots; ++m) {
        const double v = mine ? -c[m] * r : t[m] - c[m] * scaled;
        t[m] = m == 0 && sub == u ? (mine ? r : scaled) : v;
      }
    }
    const double first = t[0];
#pragma unroll
    for (int m = 0; m + 1 < kSlots; ++m) t[m] = t[m + 1];
    t[kSlots - 1] = first;
  }
}

// The trailing update of block k0 (none if k0 < 0), one workgroup per tile.
// The tile of the next block's pivots goes first and is inverted on the way,
// behind the other tiles' work.
// What bounds it: at 3,375 rows 91 MB read and 91 MB written per block (27 us
// at the rate of a copy of that size) beside 64 FP64 MFMA of 64 cycles per
// wave and tile (19 us); it takes 51 us. At 8,000 rows it moves 3.9 TB/s, a
// copy 4.7. All of a tile's 48 loads per thread are in flight together, and
// three workgroups fit a CU. The whole inverse takes 3.3 ms at 3,375 rows and
// 33.7 at 8,000; with a load at a time per thread and four launches a block it
// took 10.8 and 91.7.
__global__ void __launch_bounds__(kBlock, 3) k_gj_update(int n, int k0, double* __restrict__ a) {
  __shared__ __align__(16) double L[kGjBlock * kGjStride];
  const int tiles = (n + kGjBlock - 1) / kGjBlock, block = k0 < 0 ? -1 : k0 / kGjBlock, next = block + 1;
  // Tile number `first` and tile 0 change places.
  const int first = next * tiles + next;
  int tile = int(blockIdx.x);
  if (next < tiles) tile = tile == 0 ? first : tile == first ? 0 : tile;
  const int ti = tile / tiles, tj = tile % tiles;
  if (ti == block || tj == block) return;
  const int i0 = ti * kGjBlock, j0 = tj * kGjBlock;
  const int rows = min(kGjBlock, n - i0), cols = min(kGjBlock, n - j0);
  double c[kSlots];
  if (k0 >= 0) {
    double l[kSlots], r[kSlots], product[kSlots];
    const int b = min(kGjBlock, n - k0);
    load_rows(l, a, n, i0, k0, rows, b);
    load_slots(r, a, n, k0, j0, b, cols);
    load_slots(c, a, n, i0, j0, rows, cols);
    stage_rows(L, l);
    __syncthreads();
    tile_product(L, r, product);
#pragma unroll
    for (int m = 0; m < kSlots; ++m) c[m] -= product[m];
  } else {
    load_slots(c, a, n, i0, j0, rows, cols);
  }
  if (ti == next && tj == next) {
    __syncthreads();
    invert_slots(c, rows, L);
  }
  store_slots(c, a, n, i0, j0, rows, cols);
}

// Between the updates of two blocks: the column panel of block k0 (none if
// k0 < 0), A_IK = -A_IK P (blockIdx.y 0), and the row panel of the next block
// K' (none after the last), A_K'J = P' A_K'J (blockIdx.y 1). The one tile that
// both panels share, A_K'K, takes both steps in the second.
__global__ void __launch_bounds__(kBlock, 3) k_gj_panels(int n, int k0, double* __restrict__ a) {
  __shared__ __align__(16) double L[kGjBlock * kGjStride];
  const int block = k0 < 0 ? -1 : k0 / kGjBlock, next = block + 1, t = int(blockIdx.x), t0 = t * kGjBlock;
  const int k1 = next * kGjBlock, b0 = k0 < 0 ? 0 : min(kGjBlock, n - k0), b1 = min(kGjBlock, n - k1);
  const int extent = min(kGjBlock, n - t0);
  double l[kSlots], r[kSlots], v[kSlots];
  if (blockIdx.y == 0) {
    if (k0 < 0 || t == block || t == next) return;
    load_rows(l, a, n, t0, k0, extent, b0);
    load_slots(r, a, n, k0, k0, b0, b0);
    stage_rows(L, l);
    __syncthreads();
    tile_product(L, r, v);
#pragma unroll
    for (int m = 0; m < kSlots; ++m) v[m] = -v[m];
    store_slots(v, a, n, t0, k0, extent, b0);
    return;
  }
  if (b1 <= 0 || t == next) return;
  double p[kSlots];
  load_rows(p, a, n, k1, k1, b1, b1);
  if (t == block) {
    load_rows(l, a, n, k1, k0, b1, b0);
    load_slots(r, a, n, k0, k0, b0, b0);
    stage_rows(L, l);
    __syncthreads();
    tile_product(L, r, v);
    // The MFMA's right factor has slot s's row in s: the accumulator's layout.
#pragma unroll
    for (int m = 0; m < kSlots; ++m) r[m] = -v[m];
    __syncthreads();
  } else {
    load_slots(r, a, n, k1, t0, b1, extent);
  }
  stage_rows(L, p);
  __syncthreads();
  tile_product(L, r, v);
  store_slots(v, a, n, k1, t0, b1, extent);
}

// x = inverse b in FP64, rounded to FP32; one workgroup per row.
__global__ void __launch_bounds__(kBlock) k_dense_apply(int n, const double* __restrict__ inverse,
    const float* __restrict__ b, float* __restrict__ x, const int* __restrict__ status) {
  if (status[0] != 0) return;
  const int i = int(blockIdx.x);
  double v = 0.0;
  for (int j = threadIdx.x; j < n; j += kBlock) v += inverse[long(i) * n + j] * double(b[j]);
  __shared__ double lds[kBlock / 64];
  v = block_sum(v, lds);
  if (threadIdx.x == 0) x[i] = float(v);
}

#define KB(k) static_cast<const int*>(buf(a, k))
#define KCF(k) static_cast<const float*>(buf(a, k))
#define KD(k) static_cast<double*>(buf(a, k))

// rows, cols, values, inverse, scratch (n = rows of the dense operator;
// inverse n*n doubles; scratch is not used): the dense inverse of the CSR
// operator, left in `inverse`.
void l_dense_invert(kh_device* d, int n, const kh_arg* a) {
  if (n > 8192) throw std::runtime_error("dense_invert: at most 8192 rows");
  if (n < 1) return;
  const long count = long(n) * n;
  double* m = KD(3);
  k_dense_clear<<<dim3(unsigned((count + kBlock - 1) / kBlock)), dim3(kBlock), 0, d->stream>>>(count, m);
  k_dense_scatter<<<dim3(blocks_for(n)), dim3(kBlock), 0, d->stream>>>(n, KB(0), KB(1), KCF(2), m);
  const unsigned tiles = unsigned((n + kGjBlock - 1) / kGjBlock);
  k_gj_update<<<dim3(1), dim3(kBlock), 0, d->stream>>>(n, -1, m);
  k_gj_panels<<<dim3(tiles, 2), dim3(kBlock), 0, d->stream>>>(n, -1, m);
  for (int k0 = 0; k0 < n; k0 += kGjBlock) {
    if (tiles > 1) k_gj_update<<<dim3(tiles * tiles), dim3(kBlock), 0, d->stream>>>(n, k0, m);
    k_gj_panels<<<dim3(tiles, 2), dim3(kBlock), 0, d->stream>>>(n, k0, m);
  }
}
// inverse, b, x, status
void l_dense_apply(kh_device* d, int n, const kh_arg* a) {
  k_dense_apply<<<dim3(unsigned(n)), dim3(kBlock), 0, d->stream>>>(
      n, KD(0), KCF(1), static_cast<float*>(buf(a, 2)), KB(3));
}

}  // namespace

const std::vector<KernelEntry>& dense_kernels() {
  static const std::vector<KernelEntry> table = {
      {KH_DENSE_INVERT, "dense_invert", "bbbbb", l_dense_invert},
      {KH_DENSE_APPLY, "dense_apply", "bbbb", l_dense_apply},
  };
  return table;
}

}  // namespace kh

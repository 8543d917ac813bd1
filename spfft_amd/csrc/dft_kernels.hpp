// Matrix kernels of the sparse 3D FFT (see dft_kernels.hip): one-dimensional
// DFTs of any length as products with the cosine and sine matrices on the
// matrix cores, pruned to the indices a sparse set holds. A plane kernel does
// the y and the x transform of a plane in one launch; the z kernels serve the
// lengths without fixed-length z kernels.
#pragma once

#include <hip/hip_runtime.h>

#include "fast_kernels.hpp"

namespace spfft {

// Sizes and orders shared by the kernels and the host code that lays out their
// tables. k: largest centred index of a set, min(i, n - i).
namespace dft {

constexpr int kTile = 16;  // lines and output slots of one matrix tile

__host__ __device__ constexpr int parities(int n) { return n % 2 == 0 ? 2 : 1; }
// Backward, slot q of an even length stands for the outputs {q, n/2 - q, n/2 + q,
// n - q} (types 0 to 3), of an odd length for {q, n - q}. Slot 0 of a packed
// length stands for {0, n/2, n/4, 3n/4}: that saves slot n/4, which costs a few
// instructions more per tile but a whole tile of 16 slots when 64 divides n.
__host__ __device__ constexpr bool packed_slot(int n) { return n % 64 == 0; }
__host__ __device__ constexpr int out_slots(int n) {
  return n % 2 != 0 ? (n + 1) / 2 : n / 4 + (packed_slot(n) ? 0 : 1);
}
// Rounds of a backward sum over |r| <= k: 4 values of r each, 8 of even lengths.
__host__ __device__ constexpr int out_rounds(int n, int k) {
  return ((n % 2 == 0 ? k / 2 : k) + 4) / 4;
}
// Inputs of those rounds: the r from 0 to out_span - 1.
__host__ __device__ constexpr int out_span(int n, int k) {
  return 4 * parities(n) * out_rounds(n, k);
}
// Last r of a forward line's input quads, and their rounds of 4.
__host__ __device__ constexpr int last_quad(int n) { return n % 2 == 0 ? n / 4 : (n - 1) / 2; }
__host__ __device__ constexpr int in_rounds(int n) { return last_quad(n) / 4 + 1; }

// Trig tables: slots of a row (a tile may start at any slot), entries of the
// backward and of the forward table of length n.
__host__ __device__ constexpr int table_slots(int slots) {
  return ((slots + kTile - 1) / kTile + 1) * kTile;
}
__host__ __device__ constexpr int out_row(int n) { return table_slots(out_slots(n)); }
__host__ __device__ constexpr int in_row(int n) { return table_slots(last_quad(n) + 1); }
__host__ __device__ constexpr int out_table(int n) {
  return parities(n) * out_rounds(n, n / 2) * 4 * out_row(n);
}
__host__ __device__ constexpr int in_table(int n) {
  return parities(n) * in_rounds(n) * 4 * in_row(n);
}

// Folded order of a line: storage element i of a set with |index| <= k sits at
// fold_at(i), the positive indices from 0 up and the negative ones from fold_end
// down, so that the pairs (r, n - r) of the rounds are r and fold_end - r, with
// zeros where the set holds nothing (fold_end itself always: it pairs with r = 0).
__host__ __device__ constexpr int fold_end(int n, int k) { return 2 * out_span(n, k) - 1; }
__host__ __device__ constexpr int fold_at(int n, int k, int i) {
  return 2 * i <= n ? i : fold_end(n, k) - (n - i);
}
// Columns of the backward plane tile: x folded (R2C: x = 0 .. kx).
__host__ __device__ constexpr int tile_columns(int nx, int kx, bool rc) {
  return ((rc ? out_span(nx, kx) : fold_end(nx, kx) + 1) + kTile - 1) / kTile * kTile;
}
// Line pitch of the z kernels' tile.
__host__ __device__ constexpr int z_pitch(int nz, int kz) { return fold_end(nz, kz) + 1 | 1; }

}  // namespace dft

// Sticks per workgroup of the matrix z kernels.
constexpr int kDftSticks = dft::kTile;

// The trig tables of a transform's three lengths (equal lengths share one):
// offsets and total, in 16-byte entries.
struct DftTables {
  int at[3] = {0, 0, 0};
  int total = 0;
  DftTables(int nx, int ny, int nz) {
    auto size = [](int n) { return dft::out_table(n) + dft::in_table(n); };
    total = size(nx);
    if (ny != nx) {
      at[1] = total;
      total += size(ny);
    }
    if (nz == nx || nz == ny) {
      at[2] = nz == nx ? 0 : at[1];
    } else {
      at[2] = total;
      total += size(nz);
    }
  }
};
void build_dft_tables(void* tables, int nx, int ny, int nz, hipStream_t stream);

// True when both directions' plane kernels serve the shape (kx, ky: largest
// centred indices of the set).
template <typename T>
bool dft_plane_supported(bool r2c, int nx, int ny, int kx, int ky);

// True when the backward plane kernel can also sum the sticks' values over z
// itself (sets of stick runs), so that no z kernel is needed.
template <typename T>
bool dft_values_supported(bool r2c, int nx, int ny, int nz, int kx, int ky);

// fromValues: nz for a backward launch from the values (FastArgs::in, hasRuns),
// 0 from the [z][stick] buffer.
template <typename T>
void launch_dft_xy(bool forward, int nx, int ny, int fromValues, const FastArgs<T>& a,
                   hipStream_t stream);
// kx, ky (kz below): the batch's largest.
template <typename T>
void launch_dft_xy_batch(bool forward, bool r2c, int nx, int ny, int fromValues, int kx, int ky,
                         const FastArgs<T>* batch, int ntrans, int nz, hipStream_t stream);

template <typename T>
void launch_dft_z(bool forward, int nx, int ny, const FastArgs<T>& a, hipStream_t stream);
template <typename T>
void launch_dft_z_batch(bool forward, bool r2c, int nx, int ny, int nz, int kz,
                        const FastArgs<T>* batch, const int2* map, int blocks, bool useRuns,
                        hipStream_t stream);

}  // namespace spfft

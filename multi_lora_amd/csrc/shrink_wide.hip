// Segment shrink without a K split over workgroups (gfx950): one launch, no
// split sums, no reduce.
//
// Workgroup = dense tile of 16 token rows over the whole reduction.  Its eight
// waves take the 128-byte pieces of K in turn (piece p: wave p mod 8),
// and their fp32 sums are added in LDS in wave order.  A wave loads a piece
// of its rows (x and every A block) in row order, eight neighbouring lanes to
// a row's 128 bytes, writes it to its own part of LDS and reads MFMA
// fragments from there: waves meet only once, at the sum.
//
// Row order is what makes it pay: in fragment order (lane l on row l % 16)
// every four neighbouring lanes ask for four cache lines, and a CU loads
// 30 GB/s of L2 hits this way; in row order, 60-85 GB/s measured in this
// kernel (one 1000-row prompt, 4096 -> 4096 at rank 64, shrink: 25.9 -> 11.6
// us).  It is bound by that rate: a tile reads its x rows and its adapter's
// whole A, (A blocks + 1) * 16 rows of K.  Whole calls against the split
// kernels (us, cold inputs): a prompt of 203 rows, 4096 -> 4096 at rank 16,
// 13.5 -> 11.4; 600 rows, 1024 -> 4096 at rank 64, 18.5 -> 15.2; fp32 rows 5, 17
// and 42, 1024 -> 1024 at rank 8, 16.9 -> 9.9; 7 prompts of 300 rows of K 4101 at
// rank 64, 70 -> 36; q|k|v of 256 fp32 rows at rank 32, 256 -> 88.  wide_pays
// (shrink.hip) has the line.
#include "kernels.h"
#include "loads.h"

namespace mlora {

namespace {

constexpr int kWideWaves = 8;
constexpr int kWideThreads = kWideWaves * kWave;

// Pieces in flight a wave (in registers), by the 16-row blocks a piece holds.
template <int BLOCKS>
constexpr int kWideDepth = BLOCKS <= 2 ? 4 : BLOCKS <= 5 ? 2 : 1;

// Sixteen bytes at an address that is only element-aligned.
struct __attribute__((packed, aligned(1))) Bytes16 {
  u32x4 v;
};

// Chunk of row `row` at element kk, of which `valid` elements exist.
template <class T, bool AL>
__device__ __forceinline__ u32x4 wide_chunk(const typename T::raw_t* row, int kk, int valid) {
  if constexpr (AL) {
    const u32x4 v = ld_chunk(row + (valid > 0 ? kk : 0));
    return valid > 0 ? v : zero_chunk();
  } else {
    if (valid >= T::VEC) return reinterpret_cast<const Bytes16*>(row + kk)->v;
    return load_row_chunk<T, false>(row, kk, valid);
  }
}

// The tile's sums of NB 16-row A blocks (slice-major; nbt <= NB of them are
// live), into `mid`.
template <class T, int NB, bool AL>
__device__ __forceinline__ void wide_tile(const ShrinkArgs& a, const TileRef& tr, int rank, unsigned char* lds) {
  using raw = typename T::raw_t;
  constexpr int VEC = T::VEC;
  constexpr int BLOCKS = NB + 1;  // x is the last
  constexpr int D = kWideDepth<BLOCKS>;
  constexpr int PIECE = 128 / static_cast<int>(sizeof(raw));  // elements of K
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15;
  const int g = lane >> 4;
  const int r8 = lane >> 3;
  const int c8 = lane & 7;
  const int end = tr.end;
  const int row0 = tr.start + tr.mt * 16;
  const int nb_act = (rank + 15) >> 4;
  const int nbt = a.n_slices * nb_act;
  unsigned char* mine = lds + wave * (BLOCKS * 2048);

  // Rows 8 i + r8 of every block, clamped to rows that exist.
  const raw* src[BLOCKS][2];
#pragma unroll
  for (int b = 0; b < BLOCKS; ++b)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      if (b < NB) {
        const int jj = b < nbt ? b : 0;
        const int s = jj / nb_act;
        src[b][i] = slice_a<raw>(a.slices, s, tr.slot, min((jj - s * nb_act) * 16 + 8 * i + r8, rank - 1));
      } else {
        src[b][i] = static_cast<const raw*>(a.x) + static_cast<int64_t>(min(row0 + 8 * i + r8, end - 1)) * a.x_stride;
      }
    }

  f32x4 acc[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int npieces = (a.in_dim + PIECE - 1) / PIECE;
  u32x4 v[D][BLOCKS][2];
  auto load = [&](int d, int q) {
    const int p = q * kWideWaves + wave;
    if (p >= npieces) return;
    const int kk = p * PIECE + c8 * VEC;
    const int valid = a.in_dim - kk;
    if ((p + 1) * PIECE <= a.in_dim) {
#pragma unroll
      for (int b = 0; b < BLOCKS; ++b)
#pragma unroll
        for (int i = 0; i < 2; ++i) v[d][b][i] = wide_chunk<T, AL>(src[b][i], kk, VEC);
    } else {
#pragma unroll
      for (int b = 0; b < BLOCKS; ++b)
#pragma unroll
        for (int i = 0; i < 2; ++i) v[d][b][i] = wide_chunk<T, AL>(src[b][i], kk, valid);
    }
  };
#pragma unroll
  for (int d = 0; d < D; ++d) load(d, d);
  for (int q = 0; q * kWideWaves + wave < npieces; q += D) {
#pragma unroll
    for (int u = 0; u < D; ++u) {
      if ((q + u) * kWideWaves + wave >= npieces) break;
      wave_lds_fence();  // the last piece's fragments are read
      // LDS row r of a block holds source chunk c ^ (r >> 1 & 7) at chunk c.
#pragma unroll
      for (int b = 0; b < BLOCKS; ++b)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int r = 8 * i + r8;
          *reinterpret_cast<u32x4*>(mine + b * 2048 + r * 128 + ((c8 ^ ((r >> 1) & 7)) << 4)) = v[u][b][i];
        }
      wave_lds_fence();
      __builtin_amdgcn_sched_barrier(0);
      load(u, q + u + D);
      __builtin_amdgcn_sched_barrier(0);
      auto frag = [&](int b, int h) {
        return *reinterpret_cast<const u32x4*>(mine + b * 2048 + r16 * 128 + (((h * 4 + g) ^ ((r16 >> 1) & 7)) << 4));
      };
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const u32x4 xf = frag(NB, h);
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[j] = T::mma(acc[j], frag(j, h), xf);
      }
    }
  }

  // The waves' sums, each in its wave's part of LDS, added in wave order.
  constexpr int UNITS = NB * kWave;
  static_assert(UNITS * sizeof(f32x4) <= BLOCKS * 2048, "a wave's sums fit its part");
  auto red = [&](int w) { return reinterpret_cast<f32x4*>(lds + w * (BLOCKS * 2048)); };
  wave_lds_fence();
#pragma unroll
  for (int j = 0; j < NB; ++j) red(wave)[j * kWave + lane] = acc[j];
  __syncthreads();
  raw* mid = static_cast<raw*>(a.mid);
  const bool vec4 = (a.r_max & 3) == 0 && (a.mid_stride & 3) == 0 &&
                    (reinterpret_cast<uintptr_t>(a.mid) & (4 * sizeof(raw) - 1)) == 0;
  for (int u = tid; u < UNITS; u += kWideThreads) {
    const int j = u >> 6;
    const int l = u & 63;
    const int t = row0 + (l & 15);
    if (j >= nbt || t >= end) continue;
    f32x4 sum = red(0)[u];
#pragma unroll
    for (int w = 1; w < kWideWaves; ++w) sum += red(w)[u];
    const int s = j / nb_act;
    const int n = (j - s * nb_act) * 16 + 4 * (l >> 4);
#pragma unroll
    for (int q = 0; q < 4; ++q) sum[q] = (n + q < rank) ? sum[q] : 0.f;
    raw* m = mid + static_cast<int64_t>(t) * a.mid_stride + s * a.r_max + n;
    if (vec4) {
      if (n >= a.r_max) continue;
      if constexpr (sizeof(raw) == 2) {
        uint2 w;
        w.x = T::pack2(sum[0], sum[1]);
        w.y = T::pack2(sum[2], sum[3]);
        *reinterpret_cast<uint2*>(m) = w;
      } else {
        *reinterpret_cast<f32x4*>(m) = sum;
      }
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (n + q < a.r_max) m[q] = T::from_f32(sum[q]);
    }
  }
}

// Columns of mid from `col_from` of every slice, of the tile's rows, zeroed.
template <class T>
__device__ __forceinline__ void zero_cols(const ShrinkArgs& a, int row0, int rows_here, int col_from) {
  using raw = typename T::raw_t;
  const int width = a.r_max - col_from;
  if (width <= 0) return;
  const int per_row = a.n_slices * width;
  for (int i = threadIdx.x; i < rows_here * per_row; i += kWideThreads) {
    const int r = i / per_row;
    const int c = i - r * per_row;
    const int s = c / width;
    static_cast<raw*>(a.mid)[static_cast<int64_t>(row0 + r) * a.mid_stride + s * a.r_max + col_from + (c - s * width)] =
        T::from_f32(0.f);
  }
}

// NBM: most A blocks of the call (4 or 8).  The body is compiled for several
// block counts, so a tile of a low rank loads no more than it needs.
template <class T, int NBM, bool AL>
__global__ __launch_bounds__(kWideThreads) void shrink_wide_kernel(ShrinkArgs a) {
  __shared__ __attribute__((aligned(16))) unsigned char lds[kWideWaves * (NBM + 1) * 2048];
  TileRef tr;
  if (!dense_tile(a.meta, a.rows, blockIdx.x, 16, &tr)) return;
  const int rank = slot_rank_of(a.meta, tr.slot, a.r_max, a.rank_mult);
  const int row0 = tr.start + tr.mt * 16;
  const int nb_act = (rank + 15) >> 4;
  zero_cols<T>(a, row0, min(16, tr.end - row0), nb_act * 16);
  if (rank == 0) return;
  const int nbt = a.n_slices * nb_act;
  if (nbt == 1)
    wide_tile<T, 1, AL>(a, tr, rank, lds);
  else if (nbt == 2)
    wide_tile<T, 2, AL>(a, tr, rank, lds);
  else if (nbt == 3)
    wide_tile<T, 3, AL>(a, tr, rank, lds);
  else if (NBM == 4 || nbt == 4)
    wide_tile<T, 4, AL>(a, tr, rank, lds);
  else if constexpr (NBM > 4) {
    if (nbt <= 6)
      wide_tile<T, 6, AL>(a, tr, rank, lds);
    else
      wide_tile<T, 8, AL>(a, tr, rank, lds);
  }
}

template <class T, int NBM>
hipError_t launch_al(const ShrinkArgs& args, int64_t tiles, bool aligned, hipStream_t stream) {
  const dim3 grid(static_cast<unsigned>(tiles));
  if (aligned)
    hipLaunchKernelGGL((shrink_wide_kernel<T, NBM, true>), grid, dim3(kWideThreads), 0, stream, args);
  else
    hipLaunchKernelGGL((shrink_wide_kernel<T, NBM, false>), grid, dim3(kWideThreads), 0, stream, args);
  return hipGetLastError();
}

template <class T>
hipError_t launch_t(const ShrinkPlan& p, const ShrinkArgs& args, bool aligned, hipStream_t stream) {
  const int64_t tiles = dense_tiles(args.meta.bs, p.m_tiles, args.rows, 16);
  if (tiles <= 0) return hipSuccess;
  if (!grid_fits(tiles * (kWideThreads / 256))) return hipErrorInvalidConfiguration;
  return p.nbt <= 4 ? launch_al<T, 4>(args, tiles, aligned, stream) : launch_al<T, 8>(args, tiles, aligned, stream);
}

}  // namespace

hipError_t launch_shrink_wide(const ShrinkPlan& p, const ShrinkArgs& args, int dtype, bool aligned, hipStream_t stream) {
  switch (dtype) {
    case MLORA_BF16: return launch_t<BF16>(p, args, aligned, stream);
    case MLORA_F16: return launch_t<F16>(p, args, aligned, stream);
    default: return launch_t<F32>(p, args, aligned, stream);
  }
}

}  // namespace mlora

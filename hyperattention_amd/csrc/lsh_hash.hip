// Angular LSH bucket ids: sign bits of r random projections, Gray-coded.
// Follows the definition in src/angular_lsh_triton.py:76-88 and :175-179 of the reference
// (bit_j = [x . P[:, j] > 0], bin = sum_j bit_j << j, bucket = perm[bin], perm[i] = i ^ (i >> 1)).
//
// lsh_hash_mfma_kernel: a wave projects 16 rows at a time with v_mfma_f32_16x16x32 (16 projection slots x rows,
// fp32 accumulation), reading the rows straight from HBM as MFMA operands: a stream of reads.  Built for rows of 32, 64,
// 96, 128 and 256 elements; a row of any other multiple of 8 elements runs in the next width with its missing
// elements (and the missing rows of the projection) read as zeros.  fp32 accumulation cannot decide the
// sign of a projection that nearly cancels, so a second MFMA on |x| and |P| gives sum |x_k P_kj|, which
// bounds the accumulation error of any summation order (d * 2^-23 * sum, used with a factor 2 margin;
// fp16/bf16 products are exact in fp32 and subnormal inputs are not flushed).  Whenever some
// |projection| is inside that bound, that projection of the 16 rows is recomputed in fp64 (products exact, sum exact
// to 2^-53): 2 % of the 16-row tiles on random data of 64 elements, 5 % of 128.
#include "ha_common.h"
#include "bucket_sort.h"
#include "lsh_tiles.h"

namespace {

// Tiles of 16 rows per wave: 8 KB, in two groups of tiles whose rows are in flight together, and fewer where the launch would
// not fill the chip with workgroups.  Short waves, many of them, read fastest: the projection's set-up of one runs beside the
// loads of the others.  TB/s at 32, 8, 4, 2, 1 tiles per wave (the better group size of each): 64 x 131072 rows of 128
// bytes 5.03, 5.60, 5.92, 5.78, 4.98; 64 x 32768 6.00, 6.52, 6.75, 6.43, 4.89; 128 x 65536 of 256 bytes 5.24, 5.82,
// 5.84, 6.14, 5.54; 34 x 32768 4.81, 5.91, 6.46, 6.41, 5.56; 32 x 20480 of 192 bytes 5.47, 6.14, 6.16, 5.92, 5.48.
constexpr int HASH_FULL_CHIP = 2048;  // workgroups
template <int PARTS>
constexpr int hash_group() { return PARTS <= 2 ? 2 : 1; }

// A row of up to PARTS*32 elements is PARTS k-steps of the MFMA: lane (m = lane%16, kg = lane/16) holds elements
// 32*part + 8*kg .. +7 of row m of the tile (a load instruction covers 64 bytes of 16 rows, the part's neighbour the rest
// of their lines) and of projection slot m, and gets the projections of row m on slots 4*kg .. +3.  (With the parts of a
// row as rows of the MFMA, so that a load instruction covered whole rows, the other parts had to be zeroed and the
// product repeated per part: 4 times the vector instructions at 128 elements, which bounded the launch: 40 x 16384 rows of
// 256 bytes 44.6 -> 26.8 us, 128 x 65536 463 -> 353; of 128 bytes, 64 x 131072 218 -> 181, 8 x 4096 7.8 -> 4.3.)
// Up to two tensors per launch (queries and keys of one forward): blockIdx.y + blockIdx.z * gridDim.y counts
// the (batch, head) sequences of the first tensor, then those of the second (a grid dimension holds 65535).
struct HashTensors {
  const void* x[2];
  void* out[2];        // bucket ids, (batch, heads, n) contiguous, int32 or (OUT8) one byte each
  int64_t sb[2], sh[2], sn[2];
  int heads[2];
  int seqs0;           // batch * heads of the first tensor
  int seqs;            // sequences of both tensors together
  int64_t n_read;      // rows of a sequence that exist; rows from there up to n hash as zero rows
  int64_t first[2], end[2];  // rows of every sequence whose ids are wanted
};

// GROUP tiles (1 or 2) in flight together.  ROWS_FIRST: the first rows are asked for ahead of the projection, as the compiler does not by itself
template <typename T, int PARTS, bool OUT8, int GROUP, bool ROWS_FIRST>
__global__ __launch_bounds__(256) void lsh_hash_mfma_kernel(const HashTensors ten, const T* __restrict__ proj, int64_t n,
                                                            int r, int64_t psb, int64_t psh, int d_real, int tiles) {
  // the first workgroups alone: in those that follow, which find the arguments in the caches, it cost 6 % of a long launch
  if (blockIdx.y < 8 && blockIdx.z == 0) ha_load_arguments<(int)sizeof(HashTensors) + 48>();
  typedef typename ElemTraits<T>::vec8 vec8;
  constexpr int D = PARTS * 32;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int seq = (int)(blockIdx.y + blockIdx.z * gridDim.y);
  if (seq >= ten.seqs) return;  // the last layer of the grid may be partly empty
  const int which = seq >= ten.seqs0 ? 1 : 0;
  const int bh = seq - (which ? ten.seqs0 : 0);
  const int heads = ten.heads[which];
  const int b = bh / heads, h = bh % heads;
  const T* xbase = (const T*)ten.x[which] + b * ten.sb[which] + h * ten.sh[which];
  const int64_t sn = ten.sn[which];
  const T* pbase = proj + b * psb + h * psh;
  int32_t* obase = OUT8 ? nullptr : (int32_t*)ten.out[which] + (int64_t)bh * n;
  uint8_t* obase8 = OUT8 ? (uint8_t*)ten.out[which] + (int64_t)bh * n : nullptr;
  const int m = lane & 15, kg = lane >> 4;

  const int64_t end = ten.end[which];
  const int64_t wave_row0 = ten.first[which] + ((int64_t)blockIdx.x * 4 + wave) * tiles * 16;
  // The loads of a group have no condition, so that all of them are in flight together: rows and pieces that do not
  // exist read the last row or the first piece, and are zeroed where the group is used (a condition on a load
  // made the compiler wait for it before the next one).
  int piece[PARTS];
#pragma unroll
  for (int pt = 0; pt < PARTS; ++pt) piece[pt] = pt * 32 + 8 * kg < d_real ? pt * 32 + 8 * kg : 0;
  const int64_t last_row = ten.n_read - 1;
  vec8 xf[GROUP][PARTS];
  auto load_rows = [&](int64_t row0) {
#pragma unroll
    for (int u = 0; u < GROUP; ++u) {
      const int64_t row = row0 + u * 16 + m;
      const T* x = xbase + (row < last_row ? row : last_row) * sn;
#pragma unroll
      for (int pt = 0; pt < PARTS; ++pt) xf[u][pt] = *reinterpret_cast<const vec8*>(x + piece[pt]);
    }
  };
  // the first rows are in flight while the projection is set up
  load_rows(wave_row0);
  if constexpr (ROWS_FIRST) __builtin_amdgcn_sched_barrier(0);

  // the projection matrix goes through LDS once per block
  typedef Projection<T, PARTS> P;
  __shared__ __attribute__((aligned(16))) T lds_p[16 * P::PITCH];
  P::stage(pbase, r, d_real, lds_p, threadIdx.x);
  __syncthreads();
  const P projection(lds_p, r, lane);

#pragma unroll 1
  for (int64_t row0 = wave_row0, wave_end = wave_row0 + tiles * 16; row0 < end;) {
    const bool all_exist = d_real == D && row0 + GROUP * 16 <= ten.n_read;
    if (!all_exist) {
#pragma unroll
      for (int u = 0; u < GROUP; ++u)
#pragma unroll
        for (int pt = 0; pt < PARTS; ++pt) {
          const bool exists = pt * 32 + 8 * kg < d_real && row0 + u * 16 + m <= last_row;
          xf[u][pt] = exists ? xf[u][pt] : vec8{};
        }
    }
    uint32_t nib[GROUP];
    projection_signs<T, PARTS, GROUP>(xf, projection, r, lane, nib);
    const uint32_t bucket = bucket_ids(nib[0], GROUP == 2 ? nib[GROUP - 1] : 0u, r);
    if (lane < 16 * GROUP && row0 + lane < end) {
      if (OUT8)
        obase8[row0 + lane] = (uint8_t)bucket;
      else
        obase[row0 + lane] = (int32_t)bucket;
    }
    row0 += GROUP * 16;
    if (row0 >= wave_end) break;
    load_rows(row0);
  }
}

template <typename T, int PARTS, bool OUT8>
int launch_hash_mfma(HashTensors ten, int64_t seqs, const void* proj, int64_t n, int64_t r, int64_t psb, int64_t psh,
                     int64_t d_real, hipStream_t stream) {
  ten.seqs = (int)seqs;
  for (int i = 0; i < 2; ++i)
    if (ten.end[i] <= 0) ten.end[i] = n;
  const int64_t rows = ten.end[0] - ten.first[0] > ten.end[1] - ten.first[1] ? ten.end[0] - ten.first[0] : ten.end[1] - ten.first[1];
  constexpr int GROUP = hash_group<PARTS>();
  int tiles = 2 * GROUP;
  while (tiles > 1 && (rows + 64 * tiles - 1) / (64 * tiles) * seqs < HASH_FULL_CHIP) tiles /= 2;
  const int64_t rows_per_block = 64 * tiles;
  if (ten.n_read <= 0 || ten.n_read > n) ten.n_read = n;
  const int64_t gy = seqs < 32768 ? seqs : 32768, gz = (seqs + gy - 1) / gy;
  dim3 grid((unsigned)((rows + rows_per_block - 1) / rows_per_block), (unsigned)gy, (unsigned)gz);
  // Rows from memory are worth asking for first, of those in the caches the projection is the later one.  Hash to placement, projection | rows first, us: 128
  // heads of 65536 rows of 256 bytes 396 | 389, 4 of 524288 114.3 | 113.4, 64 of 131072 of 128 bytes 227 | 225; 34 of 32768 of 256 (280 MB) 54.1 | 55.7,
  // 64 of 32768 of 128 (268 MB) 55.6 | 56.3; 32768 of 128 rows, which leave half of the waves idle, 160 | 163.5.
  const bool rows_first = rows >= 1024 && (double)rows * seqs * PARTS * 64 > 400e6;
  auto kernel = rows_first && tiles % GROUP == 0 ? lsh_hash_mfma_kernel<T, PARTS, OUT8, GROUP, true>
                : tiles % GROUP == 0             ? lsh_hash_mfma_kernel<T, PARTS, OUT8, GROUP, false>
                                                 : lsh_hash_mfma_kernel<T, PARTS, OUT8, 1, false>;
  hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream, ten, (const T*)proj, n, (int)r, psb, psh, (int)d_real, tiles);
  return ha_launch_status("ha_lsh_hash");
}

}  // namespace

extern "C" int ha_lsh_hash(const void* x, const void* proj, int32_t* buckets, int64_t batch,
                           int64_t heads, int64_t n, int64_t d, int64_t r, int64_t x_stride_b,
                           int64_t x_stride_h, int64_t x_stride_n, int64_t proj_stride_b,
                           int64_t proj_stride_h, int dtype, void* stream) {
  return ha_hash_i32(x, proj, buckets, batch, heads, n, n, d, r, x_stride_b, x_stride_h, x_stride_n, proj_stride_b,
                     proj_stride_h, dtype, (hipStream_t)stream);
}

// ha_lsh_hash for sequences of which only the first n_read rows exist: the ids of rows n_read .. n-1 are those
// of zero rows (the rows the causal recursion appends to odd lengths)
int ha_hash_i32(const void* x, const void* proj, int32_t* buckets, int64_t batch, int64_t heads, int64_t n,
                int64_t n_read, int64_t d, int64_t r, int64_t x_stride_b, int64_t x_stride_h, int64_t x_stride_n,
                int64_t proj_stride_b, int64_t proj_stride_h, int dtype, hipStream_t stream) {
  HA_REQUIRE(x && proj && buckets, HA_ERR_NULL, "ha_lsh_hash: null pointer");
  HA_REQUIRE(dtype == HA_F16 || dtype == HA_BF16, HA_ERR_DTYPE, "ha_lsh_hash: Only support fp16 and bf16");
  HA_REQUIRE(batch > 0 && heads > 0 && n > 0, HA_ERR_SHAPE, "ha_lsh_hash: batch, heads, n must be positive");
  HA_REQUIRE(batch * heads < (1ll << 30), HA_ERR_SHAPE, "ha_lsh_hash: batch*heads must be below 2^30");
  HA_REQUIRE(r >= 1, HA_ERR_SHAPE, "ha_lsh_hash: Invalid value for num_projs");
  HA_REQUIRE(r <= 16, HA_ERR_UNSUPPORTED, "ha_lsh_hash: num_projs > 16 is not supported");
  HA_REQUIRE(d >= 8 && d <= 256 && d % 8 == 0, HA_ERR_HEADDIM, "ha_lsh_hash: d must be a multiple of 8 in [8, 256]");
  HA_REQUIRE(x_stride_n % 8 == 0 && x_stride_h % 8 == 0 && x_stride_b % 8 == 0 && ((uintptr_t)x % 16) == 0,
             HA_ERR_SHAPE, "ha_lsh_hash: rows must be 16-byte aligned");
  hipStream_t s = stream;
  HashTensors ten = {};
  ten.x[0] = x; ten.out[0] = buckets;
  ten.sb[0] = x_stride_b; ten.sh[0] = x_stride_h; ten.sn[0] = x_stride_n;
  ten.heads[0] = ten.heads[1] = (int)heads;
  ten.seqs0 = (int)(batch * heads);
  ten.n_read = n_read;
  // built for rows of 32, 64, 96, 128 and 256 elements; a shorter row runs in the next width
#define HA_HASH_MFMA(DD)                                                                                              \
  if (d <= DD) {                                                                                                          \
    if (dtype == HA_F16)                                                                                                  \
      return launch_hash_mfma<f16_t, DD / 32, false>(ten, batch * heads, proj, n, r, proj_stride_b, proj_stride_h, d, s); \
    return launch_hash_mfma<bf16_t, DD / 32, false>(ten, batch * heads, proj, n, r, proj_stride_b, proj_stride_h, d, s);  \
  }
  HA_HASH_MFMA(32) HA_HASH_MFMA(64) HA_HASH_MFMA(96) HA_HASH_MFMA(128) HA_HASH_MFMA(256)
#undef HA_HASH_MFMA
  return ha_fail(HA_ERR_HEADDIM, "ha_lsh_hash: d must be a multiple of 8 in [8, 256]");
}

// Bucket ids of the queries and keys of one forward pass as one byte each (r <= 8 projections, one shared
// projection matrix), in one launch.  q: (batch, heads, n_read, d), k: (batch, kv_heads, n_read, d), d a multiple of 8 up to 128;
// ids: n >= n_read per sequence, the ids past n_read being those of zero rows.  Wanted are the queries' from row q_first
// on and the keys' before row k_end.
int ha_hash_pair_u8(const void* q, const void* k, const void* proj, uint8_t* ids_q, uint8_t* ids_k, int64_t batch,
                    int64_t heads, int64_t kv_heads, int64_t n, int64_t n_read, int64_t d, int64_t r,
                    const int64_t (&q_strides)[3], const int64_t (&k_strides)[3], int64_t q_first, int64_t k_end, int dtype,
                    hipStream_t stream) {
  HA_REQUIRE(r >= 1 && r <= 8, HA_ERR_UNSUPPORTED, "ha_forward: byte-sized bucket ids need at most 8 projections");
  HA_REQUIRE(batch * (heads + kv_heads) < (1ll << 30), HA_ERR_SHAPE, "ha_forward: batch*(heads + kv_heads) must be below 2^30");
  HashTensors ten = {};
  ten.x[0] = q; ten.x[1] = k; ten.out[0] = ids_q; ten.out[1] = ids_k;
  ten.sb[0] = q_strides[0]; ten.sh[0] = q_strides[1]; ten.sn[0] = q_strides[2];
  ten.sb[1] = k_strides[0]; ten.sh[1] = k_strides[1]; ten.sn[1] = k_strides[2];
  ten.heads[0] = (int)heads; ten.heads[1] = (int)kv_heads;
  ten.seqs0 = (int)(batch * heads);
  ten.n_read = n_read;
  ten.first[0] = q_first; ten.end[0] = n;
  ten.first[1] = 0; ten.end[1] = k_end;
  const int64_t seqs = batch * (heads + kv_heads);
#define HA_HASH_PAIR(DD)                                                                                  \
  if (d <= DD) {                                                                                               \
    if (dtype == HA_F16) return launch_hash_mfma<f16_t, DD / 32, true>(ten, seqs, proj, n, r, 0, 0, d, stream); \
    return launch_hash_mfma<bf16_t, DD / 32, true>(ten, seqs, proj, n, r, 0, 0, d, stream);                    \
  }
  HA_HASH_PAIR(32) HA_HASH_PAIR(64) HA_HASH_PAIR(96) HA_HASH_PAIR(128)
#undef HA_HASH_PAIR
  return ha_fail(HA_ERR_UNSUPPORTED, "ha_forward: paired hash not built for head dim %lld", (long long)d);
}

// Hand-written 16-bit GEMM for projections with few rows (the text stream of a dual-stream block, small images):
// interface between linear.hip (problem checks, dispatch) and gemm_bf16.hip (the kernel).
#pragma once

#include "odit_common.h"

namespace odit {

// y[M,N] = epilogue(x[M,K] W[N,K]^T); the epilogue codes are those of odit_linear.
struct GemmCall {
  const void *x, *w, *bias, *residual, *gate;
  void* out;
  int M, N, K;
  int64_t ldx, ldw, ldo, ldr;
  int epilogue;       // enum odit_epilogue
  int gate_f32;       // gate (and, in the pre-scaled form, bias) are float32
  int rows_per_gate;  // consecutive rows that share one gate vector (0 = all rows)
  int64_t ldg;        // elements between consecutive gate vectors (and pre-scaled bias vectors)
  int clip = 0;       // a gated result of f16 is held to the largest finite value (ODIT_LINEAR_CLIP)
};

constexpr int kGemmBM = 128;  // rows of x per output tile
constexpr int kGemmBN = 256;  // rows of W (output features) per output tile, at most
constexpr int kGemmBK = 64;   // reduction elements per pipeline step

// scratch of the kernel: one 64-bit ticket word per output tile, then two partial-tile slots per workgroup
constexpr size_t kGemmCounterBytes = 32768;
constexpr size_t kGemmSlotBytes = static_cast<size_t>(kGemmBM) * kGemmBN * sizeof(float);
constexpr int kGemmMaxWorkers = 256;
constexpr size_t kGemmScratchBytes = kGemmCounterBytes + 2 * kGemmMaxWorkers * kGemmSlotBytes;

// whether the kernel takes this problem (bf16 or fp16, K a multiple of 64, N of 8, 16-byte aligned rows, operands
// addressable with 32-bit byte offsets, at most 256 row tiles and 4096 output tiles)
bool gemm_streamk_takes(const GemmCall& c, int dtype);

// One problem (count 1) or two of the same N, K and epilogue in one launch (count 2).
// `scratch` (kGemmScratchBytes, 256-byte aligned): its first kGemmCounterBytes must have been zero-filled
// once; they are zero again when the kernel has finished, and what an unfinished launch left there is
// overridden by the next launch (its ticket words carry a larger epoch).
int launch_gemm_streamk(const GemmCall* c, int count, int dtype, void* scratch, hipStream_t stream);

// compute units of the current device (0 when it cannot be read)
int device_cus();

// expected time of the launch (us), 0 where the kernel has no plan for it
float gemm_streamk_us(int M0, int M1, int N, int K, int cus);

// ---- gemm_tile.h, gemm_bf16_tile.hip: output tiles of 256 x 256 or 128 x 256, for many rows -------
// whether the kernel takes this problem (bf16 or fp16, K a multiple of 64, N of 8, 8 rows or more, 16-byte aligned rows,
// operands addressable with 32-bit byte offsets)
bool gemm_tile_takes(const GemmCall& c, int dtype);

// the last K - k_split elements of every row of x come from here (k_split a multiple of 64)
struct TileX2 {
  const void* x;
  int64_t ldx;
  int k_split;
};

struct TilePlan {
  int bm = 0;             // rows per tile (0: no plan)
  int tiles0, tiles1, tiles;  // tiles of the first problem, of the first two, of all
  int whole, parts;       // tiles that are not cut along the reduction; parts of each of the others
  int grid;
  float us;               // expected time
};
// One problem, or two or three of the same K; `scratch`: whether tiles may be cut.
TilePlan plan_gemm_tile(const GemmCall* c, int count, int cus, bool scratch);

// One problem, or two or three of the same K in one launch. `scratch` as for launch_gemm_streamk, or null (no tile is cut). `x2`: with
// one problem only.
int launch_gemm_tile(const GemmCall* c, int count, const TileX2* x2, int dtype, void* scratch, hipStream_t stream);
// gemm_tile_unless.hip: one problem, and nothing where *unless (device memory) is not 0 when the launch begins
int launch_gemm_tile_unless(const GemmCall& c, const int* unless, int dtype, void* scratch, hipStream_t stream);

// gemm_tile_apart.hip: one problem, every tile whole, its epilogue in the library's order of operations
int launch_gemm_tile_apart(const GemmCall& c, int dtype, hipStream_t stream);

// Which tiles of 256 x 256 the library's kernel that is never run sums in pieces, and where it parts them, seen from what it gave for sums that lose a term
// exactly where they are parted (eight problems that it parts, 120 to 8220 tiles and 206 to 256 workers: all 1617 parted tiles as here). Its tiles are numbered in
// groups of 16 row tiles, features outer; the last workers + tiles % workers of them (of fewer tiles than workers all), from `from` on, are shared out in equal numbers
// of steps, the first `more` workers one more. A tile's sums are added in the order of their steps. share 0: every tile is whole. `known` false: a worker has no step.
struct TileShares {
  bool known;
  int tiles, from, share, more;
};
inline TileShares tile_shares(int M, int N, int K, int workers) {
  const int tiles = (M + 255) / 256 * ((N + 255) / 256);
  if (workers <= 0) return {false, tiles, tiles, 0, 0};
  if (tiles % workers == 0) return {true, tiles, tiles, 0, 0};
  const int shared = tiles % workers + (tiles > workers ? workers : 0), steps = shared * (K / 64);
  if (steps < workers) return {false, tiles, tiles, 0, 0};
  return {true, tiles, tiles - shared, steps / workers, steps % workers};
}
// gemm_tile_shared.hip: one problem, the same with these shares (known; with share > 0 it needs `scratch`)
int launch_gemm_tile_shared(const GemmCall& c, int dtype, const TileShares& shares, void* scratch, hipStream_t stream);

// whether 32 bits hold the byte offsets of so many rows
inline bool gemm_rows_fit(int rows, int64_t ld, int K) { return (static_cast<uint64_t>(rows) * ld + K) * 2 < (1ull << 32); }
// the last row that a tile's rows of padding are fetched as: their own place past the operand's end, or where those offsets would wrap around the operand's last row
inline int tile_padding_row(int rows, int tile, int64_t ld, int K) {
  const int end = (rows + tile - 1) / tile * tile;
  return gemm_rows_fit(end, ld, K) ? end : rows - 1;
}

// ---- gemm_tile_heads.hip: the tile kernel with query, key and value heads at its end -------
// Output of a projection to 3 HD features: per batch entry S rows of queries, keys and values of HD / D heads, the first two normed
// over each head (mean of squares + eps), weighted and rotated in pairs (2 i, 2 i + 1), into rows offset .. of joint tensors [B, S_total, HD].
struct HeadsOut {
  void *q, *k, *v;
  const void *wq, *wk;      // [D], of the tensors' type
  const float *cos, *sin;   // [S, D / 2]
  int S, offset, S_total, HD, D;
  uint32_t div_mul, div_shift;  // (filled in by the launch)
  float eps;
};
// beside gemm_tile_takes, of a call whose `out` is not used
bool gemm_tile_heads_takes(const GemmCall& c, const HeadsOut& h);
// One problem, or two of the same K; heads[i].q null: an ordinary output without a gate. `scratch` as for launch_gemm_tile.
int launch_gemm_tile_heads(const GemmCall* c, int count, const HeadsOut* heads, int dtype, void* scratch, hipStream_t stream);

// ---- gemm_small.hip: 64 x 64 output tiles, for products that are small altogether -------
// One problem, or two of the same N and K in one launch, which gemm_streamk_takes takes. No scratch.
bool gemm_small_rule(const GemmCall* c, int count, int cus, int max_k);
int launch_gemm_small(const GemmCall* c, int count, int dtype, hipStream_t stream);
// LayerNorm without affine and modulation of a problem's rows, x' = norm(x) (1 + scale) + shift, in front of the product: shift and scale of
// the tensors' type, one row for S rows of x, `stride` elements apart. For one problem or two of K <= kSmallNormK.
struct RowNorm {
  const void *shift, *scale;
  int64_t stride;
  int S;
  float eps;
};
constexpr int kSmallNormK = 256;
// (`heads` with two problems only)
int launch_gemm_small_norm(const GemmCall* c, int count, const RowNorm* norm, const HeadsOut* heads, int dtype, hipStream_t stream);
// two problems of the same N, the second one's rows RMS-normed and weighted (K of it 64, 128 or 256)
int launch_gemm_small_stem(const GemmCall* c, const void* weight, float eps, int dtype, hipStream_t stream);
// the same with query, key and value heads of 64 features (gemm_small_heads.hip)
int launch_gemm_small_heads(const GemmCall* c, int count, const HeadsOut* heads, int dtype, hipStream_t stream);


// ---- linear_head.hip: a norm of the rows and a projection to few features -------
// features to a tile, 0 where the kernel cannot take the problem or is not the faster way; one problem of K 1024, 2048 or 3072 and N up to 64
int linear_head_features(const GemmCall& c, const RowNorm& n, int dtype, int cus);
int launch_linear_head(const GemmCall& c, const RowNorm& n, int features, int dtype, hipStream_t stream);

}  // namespace odit

// fp32 matrix products on the bf16 matrix cores: C(m, n) = sum over k of A(m, k) B(n, k) (+ bias(n)).
//
// The projections of a layer with fp32 parameters are nine tenths of its time, and fp32 MFMA gives 157 TFLOP/s where
// bf16 MFMA gives sixteen times as much.  Each operand element is taken as the sum of three bf16 values,
//     x = x1 + x2 + x3,   x1 = bf16(x),   x2 = bf16(x - x1),   x3 = x - x1 - x2
// which hold its 24 bits exactly, whatever else is in its row, and C is accumulated in fp32 from the six products that
// fp32 can see: x1 y1, x1 y2, x2 y1, x2 y2, x1 y3, x3 y1.  The three left out are below 2^-24 of the pair's product (2^-28
// as a rule).  The leading products have an accumulator to themselves, so that the smaller ones are not rounded away
// against it one by one: K / 16 roundings of C where a chain of fp32 multiply-adds has K.  Relative error (2-norm)
// against float64, here and by the library's fp32 kernels: 9e-8 and 2.9e-7 (32768 rows, 1024 -> 4096), 3.9e-7 and 1.1e-6,
// 8.2e-7 and 3.2e-6 (its gradients); rows with 2, 4 and 16 nonzeros 2.6e-8 and 3.1e-8, 2.8e-8 and 5.1e-8, 3.3e-8 and
// 7.1e-8, with one 2.6e-8 and 2.5e-8 (0 and 0 where it is a power of two).
//
// Both operands are scaled by 2^16 on their way (and C by 2^-32 at the end), exactly: x3's last bit is 2^-149 for the
// smallest numbers, and bf16 ends at 2^-133.  What no bf16 value holds, infinities, NaN and magnitudes from 2^111 up,
// turns the tile's results into infinities or NaN, and so does an overflow on the way; such a tile is computed again with
// fp32 MFMA from the same operands, so that it ends as fp32 arithmetic does.
#include "scan_common.h"

namespace qssm {

namespace {

constexpr int kBM = kSplitTileM, kBN = kSplitTileN, kBK = 16;
constexpr int kPlaneA = kBM * kBK * 2, kPlaneB = kBN * kBK * 2;   // bytes of one bf16 plane of a stage
constexpr int kStage = 3 * (kPlaneA + kPlaneB);

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float float2v __attribute__((ext_vector_type(2)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef float float16v __attribute__((ext_vector_type(16)));

constexpr float kScale = 0x1p16f, kUnscale = 0x1p-32f;   // of an operand, of a product

// Byte offset of (row, eight k's) within a plane: 32 bytes a row, its two 16-byte halves swapped in a pattern that
// lets eight (and sixteen) neighbouring rows' accesses of one half cover all banks.
__device__ __forceinline__ int lds_at(int row, int half) {
  return row * 32 + ((half ^ (row >> 2) ^ (row >> 3)) & 1) * 16;
}

// Eight elements as bf16 parts.
struct Parts {
  bf16x8 p[3];
};

// A stage of one operand in a thread's registers: U units of eight consecutive k's of one row.
// KSTRIDED: the operand is stored [k][row] (lanes run along the rows), else [row][k].
template <bool KSTRIDED, int ROWS>
struct Fetch {
  static constexpr int U = ROWS * 2 / 256;
  float v[U][8];
  uint32_t off[U];   // byte offset of the unit from the tile's base
  int slot[U];       // where its parts go in a plane
  int kh[U];         // first k of the unit inside the stage

  __device__ __forceinline__ void place(int row0, int n_rows, int64_t ld) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int idx = (int)threadIdx.x + 256 * u;
      const int row = KSTRIDED ? idx % ROWS : idx >> 1, half = KSTRIDED ? idx / ROWS : idx & 1;
      const int r = row0 + row < n_rows ? row : n_rows - 1 - row0;   // rows past the end repeat the last one
      off[u] = KSTRIDED ? (uint32_t)((half * 8) * (int)ld + r) * 4u : (uint32_t)(r * (int)ld + half * 8) * 4u;
      slot[u] = lds_at(row, half);
      kh[u] = half * 8;
    }
  }
  // `base` points at (k0, row0); `left` = k's from k0 to the end.
  template <bool RAGGED>
  __device__ __forceinline__ void load(int u, const char* base, int64_t ld, int left) {
    if (!RAGGED || left >= kBK) {
      if constexpr (KSTRIDED) {
#pragma unroll
        for (int i = 0; i < 8; ++i) v[u][i] = *reinterpret_cast<const float*>(base + (int64_t)i * ld * 4 + off[u]);
      } else {
        const float4v lo = *reinterpret_cast<const float4v*>(base + off[u]);
        const float4v hi = *reinterpret_cast<const float4v*>(base + off[u] + 16u);
#pragma unroll
        for (int i = 0; i < 4; ++i) { v[u][i] = lo[i]; v[u][4 + i] = hi[i]; }
      }
    } else {   // the last stage of a run of k's: zeros past its end
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        v[u][i] = 0.0f;
        if (kh[u] + i < left) v[u][i] = *reinterpret_cast<const float*>(base + (KSTRIDED ? (int64_t)i * ld * 4 : i * 4) + off[u]);
      }
    }
  }
  // Elements 2 q and 2 q + 1 of a unit, scaled, as parts: every difference is exact.
  __device__ __forceinline__ void split(int u, int q, Parts& t) const {
    float2v x = {v[u][2 * q] * kScale, v[u][2 * q + 1] * kScale};
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const bf16x2 b = __builtin_convertvector(x, bf16x2);
      t.p[k][2 * q] = b[0];
      t.p[k][2 * q + 1] = b[1];
      x = float2v{x[0] - (float)b[0], x[1] - (float)b[1]};
    }
  }
  __device__ __forceinline__ void put(int u, char* planes, int plane_bytes, const Parts& t) const {
#pragma unroll
    for (int k = 0; k < 3; ++k) *reinterpret_cast<bf16x8*>(planes + k * plane_bytes + slot[u]) = t.p[k];
  }
};

// The parts of A and of B in the six products of a pair of elements, smallest first.
constexpr int kPartA[6] = {2, 0, 1, 1, 0, 0}, kPartB[6] = {0, 2, 1, 0, 1, 0};

// The product for callers without scratch and for small ones (the packed kernel's start and end are longer).
//
// Tile of 128 x 128, four wavefronts of 64 x 64 each (2 x 2 MFMA tiles of 32 x 32 in two accumulators, 128 registers),
// stages of 16 k's in two LDS buffers with one barrier per stage.  A stage's fp32 elements are in flight to registers while
// the stage before it is multiplied; they are split on their way into LDS, so no 16-bit copy of an operand exists in
// memory.  48 KB of LDS and under 256 registers: two workgroups per compute unit, one multiplying while the other waits
// or splits.  The products of a layer with 32768 rows, hidden 1024, state 4096 run at 189, 195 and 188 TFLOP/s (outputs, input
// gradient, weight gradients), six times that on the bf16 units, near the 1.2 PFLOP/s of a large bf16 product of the library
// on this card; the library's fp32 kernels reach 143 to 152.  Matrix cores busy 59 % of the cycles, at 1.8 GHz; 5.4 other
// vector instructions per product, most of them conversions, take two thirds of the issue slots beside them.
//
// RAGGED: K is no multiple of 16, so that the last stage of a run of k's is filled up with zeros; without it the loop
// over the stages has no branch and its loads, conversions and products are scheduled as one block.
template <bool AKS, bool BKS, bool RAGGED>
__global__ void __launch_bounds__(256, 2) split_gemm_kernel(const SplitGemmArgs p) {
  __shared__ __align__(16) char lds[2 * kStage];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;

  // Workgroup i runs on XCD i mod 8: every XCD gets a run of consecutive tiles, ordered in patches of eight tiles of m
  // by n, so that the workgroups of an XCD share their rows of A and B in its L2.
  const int tm = (p.M + kBM - 1) / kBM, tn1 = (p.N + kBN - 1) / kBN, tn = tn1 * p.batch;
  const int total = tm * tn * p.splits;
  const int xcd = blockIdx.x & 7, per = total >> 3, extra = total & 7;
  int id = xcd * per + (xcd < extra ? xcd : extra) + (blockIdx.x >> 3);
  const int split = id / (tm * tn);
  id -= split * (tm * tn);
  const int patch = id / (8 * tn), m_first = patch * 8;
  const int m_count = tm - m_first < 8 ? tm - m_first : 8;
  id -= patch * (8 * tn);
  const int n_tile = id / m_count;
  const int m0 = (m_first + id - n_tile * m_count) * kBM;
  const int prob = n_tile / tn1;
  const int n0 = (n_tile - prob * tn1) * kBN;

  const int stages_per = (p.K + kBK - 1) / kBK, stages = stages_per * p.segments;
  const int s_begin = (int)((int64_t)stages * split / p.splits), s_end = (int)((int64_t)stages * (split + 1) / p.splits);
  float16v acc[2][2][2];   // [0]: products of the leading parts, [1]: the smaller ones
#pragma unroll
  for (int k = 0; k < 2; ++k)
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[k][i][j][r] = 0.0f;

  const int wm = (wave >> 1) * 64, wn = (wave & 1) * 64;
  {
    int seg = s_begin / stages_per, k0 = (s_begin - seg * stages_per) * kBK;
    Fetch<AKS, kBM> fa;
    Fetch<BKS, kBN> fb;
    fa.place(m0, p.M, p.lda);
    fb.place(n0, p.N, p.ldb);
    int next = s_begin;   // the stage the next load takes; after the last one it is taken again, and never used
    const int a_step = AKS ? kBK * (int)p.lda : kBK, b_step = BKS ? kBK * (int)p.ldb : kBK;   // elements
    const float *a, *b;
    auto start_run = [&]() {
      a = p.a[p.segments > 1 ? seg : prob] + (AKS ? (int64_t)k0 * p.lda + m0 : (int64_t)m0 * p.lda + k0);
      b = p.b[p.segments > 1 ? seg : prob] + (BKS ? (int64_t)k0 * p.ldb + n0 : (int64_t)n0 * p.ldb + k0);
    };
    start_run();
    auto load_a = [&]() { fa.template load<RAGGED>(0, reinterpret_cast<const char*>(a), p.lda, p.K - k0); };
    auto load_b = [&]() { fb.template load<RAGGED>(0, reinterpret_cast<const char*>(b), p.ldb, p.K - k0); };
    auto advance = [&]() {
      if (next + 1 >= s_end) return;
      ++next;
      k0 += kBK;
      a += a_step;
      b += b_step;
      if (k0 >= p.K) {
        k0 = 0;
        ++seg;
        start_run();
      }
    };
    Parts t;
    load_a();
    load_b();
    advance();
#pragma unroll
    for (int q = 0; q < 4; ++q) fa.split(0, q, t);
    fa.put(0, lds, kPlaneA, t);
    load_a();
#pragma unroll
    for (int q = 0; q < 4; ++q) fb.split(0, q, t);
    fb.put(0, lds + 3 * kPlaneA, kPlaneB, t);
    load_b();
    advance();
    lds_barrier();
    const int frag = lds_at(lane & 31, lane >> 5);   // (rows + 32 keep the pattern)
    for (int s = s_begin; s < s_end; ++s) {
      const char* st = lds + ((s - s_begin) & 1) * kStage;
      char* other = lds + ((s + 1 - s_begin) & 1) * kStage;   // read last a stage ago: all have passed the barrier since
      bf16x8 af[3][2], bf[3][2];
#pragma unroll
      for (int k = 0; k < 3; ++k) {   // in the order the products ask for them
        const int ka = k == 0 ? 2 : k == 1 ? 0 : 1, kb = k == 0 ? 0 : k == 1 ? 2 : 1;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          af[ka][i] = *reinterpret_cast<const bf16x8*>(st + ka * kPlaneA + (wm + i * 32) * 32 + frag);
          bf[kb][i] = *reinterpret_cast<const bf16x8*>(st + 3 * kPlaneA + kb * kPlaneB + (wn + i * 32) * 32 + frag);
        }
      }
      // Products and, in their shadow, the next stage: three products, then the conversion of two elements; every twelve
      // products a unit goes into LDS and is asked for again, a whole stage before its next use.  The order is pinned:
      // left alone, all conversions move to the front, where they wait for loads that have just been issued.
#pragma unroll
      for (int n = 0; n < 24; ++n) {
        const int k = n >> 2, i = (n >> 1) & 1, j = n & 1;
        acc[k < 5][i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[kPartA[k]][i], bf[kPartB[k]][j], acc[k < 5][i][j], 0, 0, 0);
        if (n % 3 == 2) {
          const int q = n / 3;
          if (q < 4) fa.split(0, q, t);
          else fb.split(0, q - 4, t);
          if (q == 3) { fa.put(0, other, kPlaneA, t); load_a(); }
          if (q == 7) { fb.put(0, other + 3 * kPlaneA, kPlaneB, t); load_b(); }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      advance();
      lds_barrier();
    }
  }
  // ---- both accumulators together, and whether all of them are numbers ---------------------------------------------
  bool odd = false;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        acc[0][i][j][r] = (acc[0][i][j][r] + acc[1][i][j][r]) * kUnscale;
        odd = odd || !(__builtin_fabsf(acc[0][i][j][r]) <= 3.402823466e38f);
      }
  if (__syncthreads_or(odd) != 0) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[0][i][j][r] = 0.0f;
    int seg = s_begin / stages_per, k0 = (s_begin - seg * stages_per) * kBK;
    for (int s = s_begin; s < s_end; ++s) {
      const float* a = p.a[p.segments > 1 ? seg : prob];
      const float* b = p.b[p.segments > 1 ? seg : prob];
#pragma unroll 1
      for (int k = k0 + (lane >> 5); k < k0 + kBK; k += 2) {
        float av[2], bv[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          int64_t m = m0 + wm + i * 32 + (lane & 31);
          m = m < p.M ? m : p.M - 1;
          av[i] = k < p.K ? a[AKS ? (int64_t)k * p.lda + m : m * p.lda + k] : 0.0f;
          int64_t n = n0 + wn + i * 32 + (lane & 31);
          n = n < p.N ? n : p.N - 1;
          bv[i] = k < p.K ? b[BKS ? (int64_t)k * p.ldb + n : n * p.ldb + k] : 0.0f;
        }
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) acc[0][i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[i], bv[j], acc[0][i][j], 0, 0, 0);
      }
      k0 += kBK;
      if (k0 >= p.K) { k0 = 0; ++seg; }
    }
  }

  // ---- store -----------------------------------------------------------------------------------------------------
  float* c = p.splits > 1 ? p.partial + ((int64_t)split * p.batch + prob) * p.M * p.N : p.c[prob];
  const int64_t ldc = p.splits > 1 ? p.N : p.ldc;
  const float* bias = p.splits > 1 ? nullptr : p.bias[prob];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int n = n0 + wn + j * 32 + (lane & 31);
    if (n >= p.N) continue;
    const float bn = bias != nullptr ? bias[n] : 0.0f;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int row = wm + i * 32 + q * 8 + (lane >> 5) * 4;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int m = m0 + row + r;
          const float v = acc[0][i][j][q * 4 + r];
          if (m < p.M) c[(int64_t)m * ldc + n] = bias != nullptr ? v + bn : v;
        }
      }
    }
  }
}

// Sum of the partial products of a launch that splits its k's, in a fixed order, four columns per lane.
__global__ void __launch_bounds__(256) split_reduce_kernel(const SplitGemmArgs p) {
  const int64_t quads = (int64_t)p.M * p.N / 4, plane = (int64_t)p.batch * p.M * p.N;
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (t >= quads * p.batch) return;
  const int prob = (int)(t / quads);
  const int64_t at = (t - prob * quads) * 4;
  const float* src = p.partial + (int64_t)prob * p.M * p.N + at;
  float4v s = *reinterpret_cast<const float4v*>(src);
  for (int k = 1; k < p.splits; ++k) s += *reinterpret_cast<const float4v*>(src + k * plane);
  const int64_t m = at / p.N;
  const int n = (int)(at - m * p.N);
  if (p.bias[prob] != nullptr)
    for (int i = 0; i < 4; ++i) s[i] += p.bias[prob][n + i];
  *reinterpret_cast<float4v*>(p.c[prob] + m * p.ldc + n) = s;
}

// ---- with one operand packed -------------------------------------------------------------------------------------

// 16 rows x 32 k's of one part, 1 KB in the order a wavefront reads it as an MFMA operand: lane l takes row l mod 16, k's
// 8 (l / 16) to 8 (l / 16) + 7, 16 bytes at 16 l.  All LDS accesses of the kernel below are such runs of 16 bytes by lane.
constexpr int kFrag = 1024;
constexpr int kPK = kPackedStageK;
constexpr int kPlaneM = kPackedTileM / 16 * kFrag, kPlaneN = kPackedTileN / 16 * kFrag;   // bytes of one part of a stage
constexpr int kPackedStage = 3 * (kPlaneM + kPlaneN);
static_assert(3 * kPlaneN == kPackedPiece, "a tile's share of the packed operand");

typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef __attribute__((address_space(1))) const char* global_bytes;

// BYTES per lane from `base` + `off` to LDS, lane by lane from `dst` on.  As a buffer access: beside global loads into LDS
// the compiler takes every wait for LDS as one for all that is under way.
template <int BYTES>
__device__ __forceinline__ void load_to_lds(const char* base, uint32_t off, char* dst) {
  const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(base), 0, 0xffffffffu, 0x00020000);
  if constexpr (BYTES == 16) __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_ptr_t)dst, 16, off, 0, 0, 0);
  else __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_ptr_t)dst, 4, off, 0, 0, 0);
}

// Eight elements, scaled, as parts: every difference is exact.
__device__ __forceinline__ void split8(const float* v, Parts& t) {
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    float2v x = {v[2 * q] * kScale, v[2 * q + 1] * kScale};
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const bf16x2 b = __builtin_convertvector(x, bf16x2);
      t.p[k][2 * q] = b[0];
      t.p[k][2 * q + 1] = b[1];
      x = float2v{x[0] - (float)b[0], x[1] - (float)b[1]};
    }
  }
}

// The parts of a matrix in the order the product's tiles take them: [tile of 256 rows][run][stage of 32 k's][part][16 rows]
// in pieces of kFrag, zeros past the ends.  One workgroup per tile and stage: 4 bytes read and 6 written per element, once,
// where the tiles of the other operand would each convert it again (20480 x 1024 weights: 39 us before a product of 6.1 ms).
template <bool KSTRIDED>
__global__ void __launch_bounds__(256) pack_parts_kernel(const PackArgs p) {
  const int stages = p.segments * p.stages_per;
  const int64_t id = blockIdx.x;
  const int stage = (int)(id % stages);
  const int tile = (int)(id / stages), run = p.segments > 1 ? stage / p.stages_per : tile / p.tiles_per;
  const int r0 = (p.segments > 1 ? tile : tile - run * p.tiles_per) * kPackedTileN;
  const int k0 = (p.segments > 1 ? stage - run * p.stages_per : stage) * kPK;
  const float* src = p.src[run];
  char* dst = p.dst + id * kPackedPiece;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int idx = (int)threadIdx.x + 256 * u;
    const int lane = idx & 63, piece = idx >> 6;   // 16 wavefronts' worth
    const int row = KSTRIDED ? (piece & 3) * 64 + lane : piece * 16 + (lane & 15);
    const int oct = KSTRIDED ? piece >> 2 : lane >> 4;
    const int r = r0 + row, k = k0 + oct * 8;
    float v[8];
    if (!KSTRIDED && r < p.rows && k + 8 <= p.K) {
      const float4v lo = *reinterpret_cast<const float4v*>(src + (int64_t)r * p.ld + k);
      const float4v hi = *reinterpret_cast<const float4v*>(src + (int64_t)r * p.ld + k + 4);
#pragma unroll
      for (int i = 0; i < 4; ++i) { v[i] = lo[i]; v[4 + i] = hi[i]; }
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        v[i] = 0.0f;
        if (r < p.rows && k + i < p.K) v[i] = src[KSTRIDED ? (int64_t)(k + i) * p.ld + r : (int64_t)r * p.ld + k + i];
      }
    }
    Parts t;
    split8(v, t);
    char* at = dst + (row >> 4) * kFrag + oct * 256 + (row & 15) * 16;
#pragma unroll
    for (int q = 0; q < 3; ++q) *reinterpret_cast<bf16x8*>(at + q * kPlaneN) = t.p[q];
  }
}

// The product with B packed.  Tile of 128 x 256, eight wavefronts of 64 x 64 each, stages of 32 k's in two LDS buffers: B
// goes there as it is, without passing through registers; A's fp32 elements pass through them and are split on the way.
//
// What bounds it is power: at 2^35 multiply-adds and more the matrix cores are busy for 67 to 76 % of the cycles at the 1.83
// to 1.93 GHz the card then holds (59 % at 1.8 for the kernel above), and the better they are fed the lower it falls.  Hence
// everything that is not a product is made rare.  16 x 16 x 32 products take less energy than 32 x 32 x 16 ones (random
// operands, nothing else running: 2.10 against 1.85 PFLOP/s).  Splitting the smaller operand once, ahead, leaves one vector
// instruction per product where there were 5.4.  A wavefront reads 24 KB of LDS for 96 products.  32768 rows, 1024 -> 4096
// five times: 189, 192 and 188 TFLOP/s -> 224, 244 and 244 (outputs, input gradient, weight gradients; the outputs' tiles
// have 32 stages only, before which and after which nothing is multiplied), six times that on the bf16 units: what the
// library's bf16 product of the same parts reaches (1456).  16384 rows, 256 -> 512 five times: 128, 134, 135 -> 153, 174, 170.
//
// A stage in the order things happen: the last 16 of a wavefront's 64 rows are multiplied after the barrier that says that
// all of this stage has been read and all of the next one is there, while the next stage's first operands are read and the
// one after it is asked for into the buffer just left.  So no wait has nothing to multiply beside it, and each load has a
// whole stage (2.2 us) to arrive.  Loads into LDS are spread between the products: six in a row hold up the wavefront that
// issues them (6 % of the launch).
//
// AKS: A is stored [k][row].  RAGGED: K is no multiple of 32.  TRANS: the result is stored [n][m] (A and B change places
// where the first operand is the one to pack).
template <bool AKS, bool RAGGED, bool TRANS>
__global__ void __launch_bounds__(512, 2) packed_gemm_kernel(const PackedGemmArgs p) {
  __shared__ __align__(16) char lds[2 * kPackedStage];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;

  // Tiles in the order of the kernel above: an XCD's workgroups share 8 tiles' rows of A and 4 tiles' rows of B in its L2.
  const int tm = (p.M + kPackedTileM - 1) / kPackedTileM, tn1 = (p.N + kPackedTileN - 1) / kPackedTileN, tn = tn1 * p.batch;
  const int total = tm * tn * p.splits;
  const int xcd = blockIdx.x & 7, per = total >> 3, extra = total & 7;
  int id = xcd * per + (xcd < extra ? xcd : extra) + (blockIdx.x >> 3);
  const int split = id / (tm * tn);
  id -= split * (tm * tn);
  const int patch = id / (8 * tn), m_first = patch * 8;
  const int m_count = tm - m_first < 8 ? tm - m_first : 8;
  id -= patch * (8 * tn);
  const int n_tile = id / m_count;
  const int m0 = (m_first + id - n_tile * m_count) * kPackedTileM;
  const int prob = n_tile / tn1;
  const int n0 = (n_tile - prob * tn1) * kPackedTileN;

  const int stages_per = (p.K + kPK - 1) / kPK, stages = stages_per * p.segments;
  const int s_begin = (int)((int64_t)stages * split / p.splits), s_end = (int)((int64_t)stages * (split + 1) / p.splits);
  float4v acc[2][4][4];   // [0]: products of the leading parts, [1]: the smaller ones
#pragma unroll
  for (int k = 0; k < 2; ++k)
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[k][i][j] = float4v{0.0f, 0.0f, 0.0f, 0.0f};

  const int wm = (wave >> 2) * 64, wn = (wave & 3) * 64;
  {
    // this lane's unit of A: 8 k's of one row
    const int arow = AKS ? tid & 127 : (wave << 4) + (lane & 15), aoct = AKS ? tid >> 7 : lane >> 4;
    const int ar = m0 + arow < p.M ? arow : p.M - 1 - m0;   // rows past the end repeat the last one
    const uint32_t aoff = AKS ? (uint32_t)(aoct * 8 * (int)p.lda + ar) * 4u : (uint32_t)(ar * (int)p.lda + aoct * 8) * 4u;
    const int aslot = (arow >> 4) * kFrag + aoct * 256 + (arow & 15) * 16;
    int seg = s_begin / stages_per, k0 = (s_begin - seg * stages_per) * kPK;
    // (picked from registers: a scalar load inside the loop would make every wait for LDS one for everything)
    const float* runs[kSplitGemmMany];
#pragma unroll
    for (int i = 0; i < kSplitGemmMany; ++i) {
      runs[i] = p.a[i];
      asm volatile("" : "+s"(runs[i]));
    }
    const float* a;
    auto start_run = [&]() {
      const int which = p.segments > 1 ? seg : prob;
      a = runs[0];
#pragma unroll
      for (int i = 1; i < kSplitGemmMany; ++i) a = which == i ? runs[i] : a;
      a += AKS ? (int64_t)k0 * p.lda + m0 : (int64_t)m0 * p.lda + k0;
    };
    start_run();
    const int64_t a_step = AKS ? (int64_t)kPK * p.lda : kPK;
    float v[8];
    auto load_a = [&]() {
      const global_bytes base = (global_bytes)a;
      const int left = p.K - k0;
      if (!RAGGED || left >= kPK) {
        if constexpr (AKS) {
#pragma unroll
          for (int i = 0; i < 8; ++i) v[i] = *(const __attribute__((address_space(1))) float*)(base + (int64_t)i * p.lda * 4 + aoff);
        } else {
          const float4v lo = *(const __attribute__((address_space(1))) float4v*)(base + aoff);
          const float4v hi = *(const __attribute__((address_space(1))) float4v*)(base + aoff + 16u);
#pragma unroll
          for (int i = 0; i < 4; ++i) { v[i] = lo[i]; v[4 + i] = hi[i]; }
        }
      } else {   // the last stage of a run of k's: zeros past its end
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          v[i] = 0.0f;
          if (aoct * 8 + i < left) v[i] = *(const __attribute__((address_space(1))) float*)(base + (AKS ? (int64_t)i * p.lda * 4 : i * 4) + aoff);
        }
        // (how many loads that were depends on the lanes, and the waits below count: none is left open here)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      }
    };
    int next = s_begin;   // the stage the next load takes; after the last one it is taken again, and never used
    auto advance = [&]() {
      if (next + 1 >= s_end) return;
      ++next;
      k0 += kPK;
      a += a_step;
      if (k0 >= p.K) {
        k0 = 0;
        ++seg;
        start_run();
      }
    };
    const int b_tile = p.segments > 1 ? n_tile : p.packed_each ? n_tile : n_tile - prob * tn1;
    const char* b = p.packed + ((int64_t)b_tile * stages + s_begin) * kPackedPiece;
    const uint32_t boff = (uint32_t)tid * 16u;
    const char* bsrc;
    const int last = s_end > s_begin ? s_end - 1 : s_begin;   // past it, it is taken again, and never used
    auto aim_b = [&](int s) { bsrc = b + (int64_t)((s < last ? s : last) - s_begin) * kPackedPiece; };
    auto load_b = [&](int i, char* st) {   // a sixth of the stage aimed at, into the stage's buffer
      load_to_lds<16>(bsrc + i * 8192, boff, st + 3 * kPlaneM + wave * 1024 + i * 8192);
    };
    auto put_a = [&](char* st, const Parts& t) {
#pragma unroll
      for (int q = 0; q < 3; ++q) *reinterpret_cast<bf16x8*>(st + q * kPlaneM + aslot) = t.p[q];
    };
    Parts t;
    bf16x8 af[2][3], bf[3][4];
    auto get_a = [&](const char* st, int i, int slot) {
#pragma unroll
      for (int q = 0; q < 3; ++q) af[slot][q] = *reinterpret_cast<const bf16x8*>(st + q * kPlaneM + ((wm >> 4) + i) * kFrag + lane * 16);
    };
    auto get_b = [&](const char* st, int q) {
#pragma unroll
      for (int j = 0; j < 4; ++j) bf[q][j] = *reinterpret_cast<const bf16x8*>(st + 3 * kPlaneM + q * kPlaneN + ((wn >> 4) + j) * kFrag + lane * 16);
    };
    auto product = [&](int i, int slot, int qa, int qb) {
      const int k = qa + qb > 0;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        acc[k][i][j] = TRANS ? __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[slot][qa], bf[qb][j], acc[k][i][j], 0, 0, 0)
                             : __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf[qb][j], af[slot][qa], acc[k][i][j], 0, 0, 0);
    };

    // Stage s_begin into the first buffer, the one after it on its way.
    char* cur = lds;
    char* oth = lds + kPackedStage;
    load_a();
    advance();
    aim_b(s_begin);
#pragma unroll
    for (int i = 0; i < 6; ++i) load_b(i, cur);
    split8(v, t);
    put_a(cur, t);
    load_a();
    advance();
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lds_barrier();
    aim_b(s_begin + 1);
#pragma unroll
    for (int i = 0; i < 6; ++i) load_b(i, oth);
    get_b(cur, 2);
    get_a(cur, 0, 0);
    get_b(cur, 1);
    for (int s = s_begin; s < s_end; ++s) {
      // 16 rows of A at a time, against all of B; the next stage's share of A is split in between.
      get_b(cur, 0);
      get_a(cur, 1, 1);
      __builtin_amdgcn_sched_barrier(0);
      product(0, 0, 0, 2);
      product(0, 0, 1, 1);
      __builtin_amdgcn_sched_barrier(0);
      split8(v, t);
      product(0, 0, 0, 1);
      product(0, 0, 2, 0);
      product(0, 0, 1, 0);
      product(0, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      put_a(oth, t);
      load_a();
      advance();
      get_a(cur, 2, 0);
      __builtin_amdgcn_sched_barrier(0);
      product(1, 1, 0, 2);
      product(1, 1, 1, 1);
      product(1, 1, 0, 1);
      product(1, 1, 2, 0);
      product(1, 1, 1, 0);
      product(1, 1, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      get_a(cur, 3, 1);
      __builtin_amdgcn_sched_barrier(0);
      product(2, 0, 0, 2);
      product(2, 0, 1, 1);
      product(2, 0, 0, 1);
      product(2, 0, 2, 0);
      product(2, 0, 1, 0);
      product(2, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      // Everything of this stage has been read, and everything of the next one is there.  (Written out: the compiler's own
      // barrier would wait for A's loads as well.)
      if constexpr (AKS) asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)\n\ts_barrier" ::: "memory");
      else asm volatile("s_waitcnt vmcnt(2) lgkmcnt(0)\n\ts_barrier" ::: "memory");
      aim_b(s + 2);
      __builtin_amdgcn_sched_barrier(0);
      load_b(0, cur);
      product(3, 1, 0, 2);
      get_b(oth, 2);
      get_a(oth, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      load_b(1, cur);
      product(3, 1, 1, 1);
      __builtin_amdgcn_sched_barrier(0);
      load_b(2, cur);
      product(3, 1, 0, 1);
      get_b(oth, 1);
      __builtin_amdgcn_sched_barrier(0);
      load_b(3, cur);
      product(3, 1, 2, 0);
      __builtin_amdgcn_sched_barrier(0);
      load_b(4, cur);
      product(3, 1, 1, 0);
      __builtin_amdgcn_sched_barrier(0);
      load_b(5, cur);
      product(3, 1, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      char* x = cur;
      cur = oth;
      oth = x;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // no load into LDS outlives the workgroup
  }
  // ---- both accumulators together, and whether all of them are numbers ---------------------------------------------
  bool odd = false;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        acc[0][i][j][r] = (acc[0][i][j][r] + acc[1][i][j][r]) * kUnscale;
        odd = odd || !(__builtin_fabsf(acc[0][i][j][r]) <= 3.402823466e38f);
      }
  // (a wavefront for itself: what follows has no barrier)
  if (__any(odd)) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[0][i][j] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
    int seg = s_begin / stages_per, k0 = (s_begin - seg * stages_per) * kPK;
    for (int s = s_begin; s < s_end; ++s) {
      const float* a = p.a[p.segments > 1 ? seg : prob];
      const float* b = p.b[p.segments > 1 ? seg : prob];
#pragma unroll 1
      for (int k = k0 + (lane >> 4); k < k0 + kPK; k += 4) {
        float av[4], bv[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          int64_t m = m0 + wm + i * 16 + (lane & 15);
          m = m < p.M ? m : p.M - 1;
          av[i] = k < p.K ? a[AKS ? (int64_t)k * p.lda + m : m * p.lda + k] : 0.0f;
          int64_t n = n0 + wn + i * 16 + (lane & 15);
          n = n < p.N ? n : p.N - 1;
          bv[i] = k < p.K ? b[p.b_kstrided ? (int64_t)k * p.ldb + n : n * p.ldb + k] : 0.0f;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            acc[0][i][j] = TRANS ? __builtin_amdgcn_mfma_f32_16x16x4f32(av[i], bv[j], acc[0][i][j], 0, 0, 0)
                                 : __builtin_amdgcn_mfma_f32_16x16x4f32(bv[j], av[i], acc[0][i][j], 0, 0, 0);
      }
      k0 += kPK;
      if (k0 >= p.K) { k0 = 0; ++seg; }
    }
  }

  // ---- store: a lane has four consecutive columns of one row of C (rows are n with TRANS) ----------------------------
  const int rows = TRANS ? p.N : p.M, cols = TRANS ? p.M : p.N;
  float* c = p.splits > 1 ? p.partial + ((int64_t)split * p.batch + prob) * p.M * p.N : p.c[prob];
  const int64_t ldc = p.splits > 1 ? cols : p.ldc;
  const float* bias = p.splits > 1 ? nullptr : p.bias[prob];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int mt = m0 + wm + i * 16, nt = n0 + wn + j * 16;
      const int row = (TRANS ? nt : mt) + (lane & 15), col = (TRANS ? mt : nt) + (lane >> 4) * 4;
      if (row >= rows || col >= cols) continue;
      float4v v = acc[0][i][j];
      if (bias != nullptr) {
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] += bias[col + r];
      }
      *reinterpret_cast<float4v*>(c + (int64_t)row * ldc + col) = v;
    }
}

}  // namespace

int64_t split_gemm_tiles(int64_t M, int64_t N, int64_t batch) {
  return ((M + kBM - 1) / kBM) * ((N + kBN - 1) / kBN) * batch;
}
static void reduce_parts(const SplitGemmArgs& p, hipStream_t stream) {
  const int64_t lanes = (int64_t)p.M * p.N / 4 * p.batch;
  hipLaunchKernelGGL(split_reduce_kernel, dim3((unsigned)((lanes + 255) / 256)), dim3(256), 0, stream, p);
}
int64_t split_gemm_stages(int64_t K, int64_t segments) { return (K + kBK - 1) / kBK * segments; }

bool launch_split_gemm(const SplitGemmArgs& p, bool a_kstrided, bool b_kstrided, hipStream_t stream) {
  const dim3 grid((unsigned)(split_gemm_tiles(p.M, p.N, p.batch) * p.splits));
  const bool ragged = p.K % kBK != 0;
#define QSSM_SPLIT_CASE(A, B, R)                                                                         \
  if (a_kstrided == A && b_kstrided == B && ragged == R)                                                 \
    hipLaunchKernelGGL((split_gemm_kernel<A, B, R>), grid, dim3(256), 0, stream, p);
  QSSM_SPLIT_CASE(false, false, false)
  QSSM_SPLIT_CASE(false, false, true)
  QSSM_SPLIT_CASE(false, true, false)
  QSSM_SPLIT_CASE(false, true, true)
  QSSM_SPLIT_CASE(true, true, false)
  QSSM_SPLIT_CASE(true, true, true)
#undef QSSM_SPLIT_CASE
  if (a_kstrided && !b_kstrided) return false;
  if (p.splits > 1) reduce_parts(p, stream);
  return true;
}

int64_t packed_gemm_tiles(int64_t M, int64_t N, int64_t batch) {
  return ((M + kPackedTileM - 1) / kPackedTileM) * ((N + kPackedTileN - 1) / kPackedTileN) * batch;
}
int64_t packed_gemm_stages(int64_t K, int64_t segments) { return (K + kPK - 1) / kPK * segments; }
uint64_t packed_bytes(int64_t N, int64_t K, int64_t many) {
  return (uint64_t)((N + kPackedTileN - 1) / kPackedTileN) * many * packed_gemm_stages(K, 1) * (3 * kPlaneN);
}

void launch_packed_gemm(const PackedGemmArgs& p, bool a_kstrided, bool trans, hipStream_t stream) {
  PackArgs k;
  const bool each = p.segments > 1 || p.packed_each;
  for (int i = 0; i < kSplitGemmMany; ++i) k.src[i] = p.b[i];
  k.dst = p.packed;
  k.ld = p.ldb;
  k.rows = p.N;
  k.K = p.K;
  k.segments = p.segments;
  k.stages_per = (int)packed_gemm_stages(p.K, 1);
  k.tiles_per = (p.N + kPackedTileN - 1) / kPackedTileN;
  const dim3 pieces((unsigned)(k.tiles_per * (each ? (p.segments > 1 ? p.segments : p.batch) : 1) * k.stages_per));
  if (p.b_kstrided) hipLaunchKernelGGL(pack_parts_kernel<true>, pieces, dim3(256), 0, stream, k);
  else hipLaunchKernelGGL(pack_parts_kernel<false>, pieces, dim3(256), 0, stream, k);

  const dim3 grid((unsigned)(packed_gemm_tiles(p.M, p.N, p.batch) * p.splits));
  const bool ragged = p.K % kPK != 0;
#define QSSM_PACKED_CASE(A, R, T)                                                              \
  if (a_kstrided == A && ragged == R && trans == T)                                            \
    hipLaunchKernelGGL((packed_gemm_kernel<A, R, T>), grid, dim3(512), 0, stream, p);
  QSSM_PACKED_CASE(false, false, false)
  QSSM_PACKED_CASE(false, true, false)
  QSSM_PACKED_CASE(true, false, false)
  QSSM_PACKED_CASE(true, true, false)
  QSSM_PACKED_CASE(false, false, true)
  QSSM_PACKED_CASE(false, true, true)
  QSSM_PACKED_CASE(true, false, true)
  QSSM_PACKED_CASE(true, true, true)
#undef QSSM_PACKED_CASE
  if (p.splits > 1) {
    SplitGemmArgs r;
    for (int i = 0; i < kSplitGemmMany; ++i) { r.c[i] = p.c[i]; r.bias[i] = p.bias[i]; }
    r.M = trans ? p.N : p.M;
    r.N = trans ? p.M : p.N;
    r.batch = p.batch;
    r.splits = p.splits;
    r.ldc = p.ldc;
    r.partial = p.partial;
    reduce_parts(r, stream);
  }
}

}  // namespace qssm

// fp32 matrix products on the 16-bit matrix cores: C(m, n) = sum over k of A(m, k) B(n, k) (+ bias(n)).
//
// The projections of a layer with fp32 parameters are nine tenths of its time, and fp32 MFMA gives 157 TFLOP/s where
// fp16 MFMA gives sixteen times as much.  Each operand element is taken as the sum of two fp16 values,
//     x * 2^e = hi + lo,   hi = fp16(x * 2^e),   lo = fp16(x * 2^e - hi)
// (22 to 24 significant bits), and C is accumulated in fp32 from three products, hi*hi + hi*lo + lo*hi.  e is chosen
// per row of A and of B from the largest magnitude in the row (amax_kernel), which puts that one just below 2^15: an
// element keeps all of its bits down to 2^-15 of its row's largest, and below that an absolute error of 2^-39 of it.
// The scales are powers of two and leave again, exactly, in the epilogue.  The left-out lo*lo and the rounding of lo
// are 2^-24 of a product each, with random signs; what an fp32 chain over k loses grows with the chain instead.
//
// A tile whose rows hold an infinity or a NaN is computed with fp32 MFMA from the same operands, so that they reach
// the result as they do in fp32 arithmetic.
#include "scan_common.h"

namespace qssm {

namespace {

constexpr int kBM = kSplitTileM, kBN = kSplitTileN, kBK = 16;
constexpr int kPlaneA = kBM * kBK * 2, kPlaneB = kBN * kBK * 2;   // bytes of one fp16 plane of a stage
constexpr int kStage = 2 * (kPlaneA + kPlaneB);
constexpr unsigned kInfBits = 0x7f800000u;

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float float2v __attribute__((ext_vector_type(2)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef float float16v __attribute__((ext_vector_type(16)));
typedef unsigned uint4v __attribute__((ext_vector_type(4)));

// Exponent that brings a row's largest magnitude into [2^14, 2^15).
__device__ __forceinline__ int scale_exp(unsigned amax_bits) {
  int e = (int)(amax_bits >> 23) - 127;
  e = e < -100 ? -100 : e;
  return 14 - e;
}
__device__ __forceinline__ float exp2_int(int e) { return __uint_as_float((unsigned)(e + 127) << 23); }

// Byte offset of (row, eight k's) within a plane: 32 bytes a row, its two 16-byte halves swapped in a pattern that
// lets eight (and sixteen) neighbouring rows' accesses of one half cover all banks.
__device__ __forceinline__ int lds_at(int row, int half) {
  return row * 32 + ((half ^ (row >> 2) ^ (row >> 3)) & 1) * 16;
}

// A stage of one operand in a thread's registers: U units of eight consecutive k's of one row.
// KSTRIDED: the operand is stored [k][row] (lanes run along the rows), else [row][k].
template <bool KSTRIDED, int ROWS>
struct Fetch {
  static constexpr int U = ROWS * 2 / 256;
  float v[U][8];
  uint32_t off[U];   // byte offset of the unit from the tile's base
  float scale[U];
  int slot[U];       // where its halves go in a plane
  int kh[U];         // first k of the unit inside the stage

  __device__ __forceinline__ void place(int row0, int n_rows, int64_t ld, const int* exps) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int idx = (int)threadIdx.x + 256 * u;
      const int row = KSTRIDED ? idx % ROWS : idx >> 1, half = KSTRIDED ? idx / ROWS : idx & 1;
      const int r = row0 + row < n_rows ? row : n_rows - 1 - row0;   // rows past the end repeat the last one
      off[u] = KSTRIDED ? (uint32_t)((half * 8) * (int)ld + r) * 4u : (uint32_t)(r * (int)ld + half * 8) * 4u;
      slot[u] = lds_at(row, half);
      kh[u] = half * 8;
      scale[u] = exp2_int(exps[row]);
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
  // Elements 2 q and 2 q + 1 of a unit as halves.
  __device__ __forceinline__ void split(int u, int q, half8& h, half8& l) const {
    const float x0 = v[u][2 * q], x1 = v[u][2 * q + 1];
    const float2v t = {x0 * scale[u], x1 * scale[u]};
    const half2v hp = __builtin_convertvector(t, half2v);
    // exact either way (the scale is a power of two); as a multiply-add it is one mixed-precision instruction
    const float2v r = {fmaf(x0, scale[u], -(float)hp[0]), fmaf(x1, scale[u], -(float)hp[1])};
    const half2v lp = __builtin_convertvector(r, half2v);
    h[2 * q] = hp[0]; h[2 * q + 1] = hp[1];
    l[2 * q] = lp[0]; l[2 * q + 1] = lp[1];
  }
  __device__ __forceinline__ void put(int u, char* hi_plane, char* lo_plane, const half8& h, const half8& l) const {
    *reinterpret_cast<half8*>(hi_plane + slot[u]) = h;
    *reinterpret_cast<half8*>(lo_plane + slot[u]) = l;
  }
};

// Tile of 256 x 128, four wavefronts of 128 x 64 each (4 x 2 MFMA tiles of 32 x 32, 128 accumulator registers), stages
// of 16 k's in two LDS buffers with one barrier per stage.  A stage's fp32 elements are in flight to registers while
// the stage before it is multiplied; they are split on their way into LDS, so no 16-bit copy of an operand exists in
// memory.  48 KB of LDS and under 256 registers: two workgroups per compute unit, one multiplying while the other waits
// or splits.  Bound by the matrix cores and what the conversions take of their issue slots: the products of a layer with
// 32768 rows, hidden 1024, state 4096 run at 310 (outputs), 350 (input gradient) and 330 TFLOP/s (weight gradients), three
// times that on the fp16 units, where the library's fp32 kernels reach 143 to 153.
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
  float16v acc[4][2];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

  const int wm = (wave >> 1) * 128, wn = (wave & 1) * 64;
  // Exponents of the tile's 256 rows of A and 128 rows of B, from the parts of their maxima (rows past the end have the
  // last one's).
  __shared__ int exps[kBM + kBN];
  auto largest = [](const unsigned* words, int parts, int64_t stride) {
    unsigned m = 0;
#pragma unroll 16
    for (int k = 0; k < parts; ++k) {
      const unsigned w = words[k * stride];
      m = m > w ? m : w;
    }
    return m;
  };
  const unsigned amax_a = largest(p.amax_a[prob] + (m0 + tid < p.M ? m0 + tid : p.M - 1), p.parts_a, p.M);
  exps[tid] = scale_exp(amax_a);
  bool odd = amax_a >= kInfBits;
  if (tid < kBN) {
    const unsigned amax_b = largest(p.amax_b[prob] + (n0 + tid < p.N ? n0 + tid : p.N - 1), p.parts_b, p.N);
    exps[kBM + tid] = scale_exp(amax_b);
    odd = odd || amax_b >= kInfBits;
  }
  const bool special = __syncthreads_or(odd) != 0;

  // where the operands of a stage start
  int seg = s_begin / stages_per, k0 = (s_begin - seg * stages_per) * kBK;
  if (!special) {
    Fetch<AKS, kBM> fa;
    Fetch<BKS, kBN> fb;
    fa.place(m0, p.M, p.lda, exps);
    fb.place(n0, p.N, p.ldb, exps + kBM);
    int next = s_begin;   // the stage the next load takes; after the last one it is taken again, and never used
    const int a_step = AKS ? kBK * (int)p.lda : kBK, b_step = BKS ? kBK * (int)p.ldb : kBK;   // elements
    const float *a, *b;
    auto start_run = [&]() {
      a = p.a[p.segments > 1 ? seg : prob] + (AKS ? (int64_t)k0 * p.lda + m0 : (int64_t)m0 * p.lda + k0);
      b = p.b[p.segments > 1 ? seg : prob] + (BKS ? (int64_t)k0 * p.ldb + n0 : (int64_t)n0 * p.ldb + k0);
    };
    start_run();
    auto load_a = [&](int u) { fa.template load<RAGGED>(u, reinterpret_cast<const char*>(a), p.lda, p.K - k0); };
    auto load_b = [&](int u) { fb.template load<RAGGED>(u, reinterpret_cast<const char*>(b), p.ldb, p.K - k0); };
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
    // Unit u of A (0, 1) or B (2) into LDS as halves, and asked for again.
    half8 h, l;
    auto split = [&](int u, int q) {
      if (u < 2) fa.split(u, q, h, l);
      else fb.split(0, q, h, l);
    };
    auto put_and_load = [&](int u, char* st) {
      if (u < 2) {
        fa.put(u, st, st + kPlaneA, h, l);
        load_a(u);
      } else {
        fb.put(0, st + 2 * kPlaneA, st + 2 * kPlaneA + kPlaneB, h, l);
        load_b(0);
      }
    };
    load_a(0);
    load_a(1);
    load_b(0);
    advance();
#pragma unroll
    for (int u = 0; u < 3; ++u) {
#pragma unroll
      for (int q = 0; q < 4; ++q) split(u, q);
      put_and_load(u, lds);
    }
    advance();
    lds_barrier();
    const int frag = lds_at(lane & 31, lane >> 5);   // (rows + 32 keep the pattern)
    for (int s = s_begin; s < s_end; ++s) {
      const char* st = lds + ((s - s_begin) & 1) * kStage;
      char* other = lds + ((s + 1 - s_begin) & 1) * kStage;   // read last a stage ago: all have passed the barrier since
      half8 ah[4], al[4], bh[2], bl[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) bh[j] = *reinterpret_cast<const half8*>(st + 2 * kPlaneA + (wn + j * 32) * 32 + frag);
#pragma unroll
      for (int i = 0; i < 4; ++i) ah[i] = *reinterpret_cast<const half8*>(st + (wm + i * 32) * 32 + frag);
#pragma unroll
      for (int j = 0; j < 2; ++j) bl[j] = *reinterpret_cast<const half8*>(st + 2 * kPlaneA + kPlaneB + (wn + j * 32) * 32 + frag);
#pragma unroll
      for (int i = 0; i < 4; ++i) al[i] = *reinterpret_cast<const half8*>(st + kPlaneA + (wm + i * 32) * 32 + frag);
      // Products and, in their shadow, the next stage: two products, then the conversion of two elements; every eight
      // products a unit goes into LDS and is asked for again, a whole stage before its next use.  The order is pinned:
      // left alone, all conversions move to the front, where they wait for loads that have just been issued.
#pragma unroll
      for (int n = 0; n < 24; ++n) {
        const int i = (n & 7) >> 1, j = n & 1;
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(n < 16 ? ah[i] : al[i], n >= 8 && n < 16 ? bl[j] : bh[j], acc[i][j], 0, 0, 0);
        if (n & 1) {
          split(n >> 3, (n & 7) >> 1);
          if ((n & 7) == 7) put_and_load(n >> 3, other);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      advance();
      lds_barrier();
    }
  } else {
    for (int s = s_begin; s < s_end; ++s) {
      const float* a = p.a[p.segments > 1 ? seg : prob];
      const float* b = p.b[p.segments > 1 ? seg : prob];
#pragma unroll 1
      for (int k = k0 + (lane >> 5); k < k0 + kBK; k += 2) {
        float av[4], bv[2];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          int64_t m = m0 + wm + i * 32 + (lane & 31);
          m = m < p.M ? m : p.M - 1;
          av[i] = k < p.K ? a[AKS ? (int64_t)k * p.lda + m : m * p.lda + k] : 0.0f;
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          int64_t n = n0 + wn + j * 32 + (lane & 31);
          n = n < p.N ? n : p.N - 1;
          bv[j] = k < p.K ? b[BKS ? (int64_t)k * p.ldb + n : n * p.ldb + k] : 0.0f;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[i], bv[j], acc[i][j], 0, 0, 0);
      }
      k0 += kBK;
      if (k0 >= p.K) { k0 = 0; ++seg; }
    }
  }

  // ---- take the scales off and store ---------------------------------------------------------------------------
  float* c = p.splits > 1 ? p.partial + ((int64_t)split * p.batch + prob) * p.M * p.N : p.c[prob];
  const int64_t ldc = p.splits > 1 ? p.N : p.ldc;
  const float* bias = p.splits > 1 ? nullptr : p.bias[prob];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int n = n0 + wn + j * 32 + (lane & 31);
    if (n >= p.N) continue;
    const int eb = exps[kBM + wn + j * 32 + (lane & 31)];
    const float bn = bias != nullptr ? bias[n] : 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int row = wm + i * 32 + q * 8 + (lane >> 5) * 4;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int m = m0 + row + r;
          const float v = special ? acc[i][j][q * 4 + r] : ldexpf(acc[i][j][q * 4 + r], -(exps[row + r] + eb));
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

// Largest magnitude (as the bits of its absolute value, which order like integers, NaN above infinity) of the rows and
// columns of a block of one of the matrices.  A workgroup takes `block_rows` rows of 256 * Q columns, a quarter of the
// rows per wavefront; its columns' maxima stay in registers over the rows.  Every block writes words of its own, and the
// product that reads them takes the largest: no atomics and nothing to clear beforehand.  Bound by memory: sixteen 16-byte
// loads per lane are in flight.
template <int Q>
__device__ __forceinline__ void amax_block(const AmaxMatrix& x, int block, unsigned (*cols_lds)[1024]) {
  constexpr int RU = 16 / Q;   // rows at a time
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int cb = block % x.col_blocks, rb = block / x.col_blocks;
  const int c0 = cb * (256 * Q);
  const int per_wave = x.block_rows / 4;   // a multiple of 16
  const int64_t r0 = (int64_t)rb * x.block_rows + wave * per_wave;
  uint4v cm[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) cm[q] = (uint4v)(0u);
  for (int k = 0; k < per_wave; k += RU) {
    if (r0 + k >= x.rows) break;
    uint4v v[RU][Q];
#pragma unroll
    for (int i = 0; i < RU; ++i) {
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const int c = c0 + q * 256 + lane * 4;
        v[i][q] = (uint4v)(0u);
        if (c < x.cols && r0 + k + i < x.rows) v[i][q] = *reinterpret_cast<const uint4v*>(x.x + (r0 + k + i) * x.ld + c);
      }
    }
    unsigned mine = 0;
#pragma unroll
    for (int i = 0; i < RU; ++i) {
      unsigned rm = 0;
#pragma unroll
      for (int q = 0; q < Q; ++q) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const unsigned m = v[i][q][e] & 0x7fffffffu;
          cm[q][e] = cm[q][e] > m ? cm[q][e] : m;
          rm = rm > m ? rm : m;
        }
      }
      if (x.row != nullptr) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
          const unsigned other = (unsigned)__shfl_xor((int)rm, o, 64);
          rm = rm > other ? rm : other;
        }
        if (lane == i) mine = rm;
      }
    }
    if (x.row != nullptr && lane < RU && r0 + k + lane < x.rows) x.row[(int64_t)cb * x.rows + r0 + k + lane] = mine;
  }
  if (x.col == nullptr) return;
#pragma unroll
  for (int q = 0; q < Q; ++q) *reinterpret_cast<uint4v*>(&cols_lds[wave][q * 256 + lane * 4]) = cm[q];
  __syncthreads();
  for (int c = threadIdx.x; c < 256 * Q && c0 + c < x.cols; c += 256) {
    unsigned m = cols_lds[0][c];
#pragma unroll
    for (int w = 1; w < 4; ++w) m = m > cols_lds[w][c] ? m : cols_lds[w][c];
    x.col[(int64_t)rb * x.cols + c0 + c] = m;
  }
}

__global__ void __launch_bounds__(256) amax_kernel(const AmaxArgs p) {
  __shared__ __align__(16) unsigned cols_lds[4][1024];
  int block = blockIdx.x, k = 0;
  while (block >= p.m[k].blocks) block -= p.m[k++].blocks;   // the grid has as many workgroups as all matrices have blocks
  if (p.m[k].wide) amax_block<4>(p.m[k], block, cols_lds);
  else amax_block<1>(p.m[k], block, cols_lds);
}

}  // namespace

int64_t split_gemm_tiles(int64_t M, int64_t N, int64_t batch) {
  return ((M + kBM - 1) / kBM) * ((N + kBN - 1) / kBN) * batch;
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
  if (p.splits > 1) {
    const int64_t lanes = (int64_t)p.M * p.N / 4 * p.batch;
    hipLaunchKernelGGL(split_reduce_kernel, dim3((unsigned)((lanes + 255) / 256)), dim3(256), 0, stream, p);
  }
  return true;
}

// Blocks of 256 columns, or 1024 where that would make more than 32 of them, and of at least 128 rows, at most 64 of
// those: few enough words for a product to look through before it starts, and a few hundred workgroups for every matrix
// that is worth the launch.
void amax_shape(int64_t rows, int cols, AmaxMatrix* m) {
  m->wide = cols > 2048 && (cols > 8192 || rows >= 16384);
  const int width = m->wide ? 1024 : 256;
  m->col_blocks = (cols + width - 1) / width;
  const int64_t per = rows < 128 * 64 ? 128 : (rows + 63) / 64;
  m->block_rows = (int)((per + 63) / 64 * 64);
  m->row_blocks = (int)((rows + m->block_rows - 1) / m->block_rows);
  m->blocks = m->row_blocks * m->col_blocks;
}

void launch_amax(const AmaxArgs& p, int count, hipStream_t stream) {
  int64_t blocks = 0;
  for (int i = 0; i < count; ++i) blocks += p.m[i].blocks;
  hipLaunchKernelGGL(amax_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, p);
}

}  // namespace qssm

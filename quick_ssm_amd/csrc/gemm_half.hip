// Weight gradients of layers whose parameters are stored in 16 bits: C(m, n) = sum over k of A[k][m] B[k][n], fp32
// accumulation, one rounding.  A is the gradient of a linear map's outputs, B its inputs, k their rows.
#include <type_traits>

#include "scan_common.h"

namespace qssm {

namespace {

constexpr int kTile = kHalfTile, kBK = kHalfStageK;
constexpr int kPlane = kTile * kBK * 2;    // bytes of a stage of one operand
constexpr int kStage = 2 * kPlane;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef short short4v __attribute__((ext_vector_type(4)));
typedef short short8v __attribute__((ext_vector_type(8)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef unsigned int uint2v __attribute__((ext_vector_type(2)));
typedef unsigned int uint4v __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef __attribute__((address_space(3))) short4v* lds_short4_t;

template <typename T>
__device__ __forceinline__ float4v mfma(const short8v& a, const short8v& b, const float4v& c) {
  if constexpr (std::is_same<T, bf16_t>::value)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

// A stage of an operand in LDS: 64 k's of 512 bytes (256 columns).  The sixteen 32-byte pieces of a k (16 columns each, what
// a 16 x 16 x 32 product takes) change places by k, so that the 16 k's which one transposing read takes of a piece lie in
// different banks.
__device__ __forceinline__ int order(int k) { return (k & 3) | ((k >> 3) & 1) << 2; }

// Sixteen columns x 32 k's as an MFMA operand: lane l gets k's 8 (l / 16) to 8 (l / 16) + 7 of column l mod 16.  A transposing
// read hands each 16 lanes four k's of 32 bytes.  (restrict, so that the compiler does not take it for a read of what loads
// into LDS are about to write, and wait for those.)
__device__ __forceinline__ short8v read_across(const char* __restrict p) {
  const short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_t)p);
  const short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_t)(p + 4 * 512));
  return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}

struct Place {
  int tile, m0, n0;   // the workgroup's tile and its first row and column of C
};
// An XCD's workgroups share the columns of 8 tiles of m and of a few of n in its L2.
__device__ __forceinline__ Place place(const HalfGemmArgs& p, int tile) {
  const int tm = (p.M + kTile - 1) / kTile, tn = (p.N + kTile - 1) / kTile;
  const int patch = tile / (8 * tn), m_first = patch * 8;
  const int m_count = tm - m_first < 8 ? tm - m_first : 8;
  const int in_patch = tile - patch * (8 * tn);
  const int n_tile = in_patch / m_count;
  return Place{tile, (m_first + in_patch - n_tile * m_count) * kTile, n_tile * kTile};
}

// Tiles of 256 x 256, eight wavefronts of 128 x 64, stages of 64 k's in two LDS buffers that loads fill without passing
// through registers; one barrier a stage, with a quarter of the stage's products behind it, as in the packed fp32 product
// (gemm_split.hip).  Both operands lie in memory k by k, and a product wants eight k's of a column in a register: the
// transposing reads turn them round on the way out of LDS.
//
// What bounds it are those reads: 155 bytes a nanosecond and compute unit by themselves (a probe; 70 a clock), 192 KB a stage
// beside 2048 cycles of products.  8192^3: 840 to 889 us, the library's 905 to 942, its product of rows in k's order 682 to
// 764.  Tried: four wavefronts of 128 x 128, a third fewer reads but one wavefront a SIMD, 872; four buffers of 32 k's, loads
// asked for three stages ahead, 889; whole rows read 16 bytes at a time and turned round by v_perm, 927.
//
// What it is for are long sums into few tiles: the rows of a batch are k here, and a weight has 4 to 320 tiles.  The tiles
// beyond full rounds of one workgroup per compute unit are dealt out in parts of their k's (qssm_weight_gradient).  16384
// rows, library -> here: 20480 x 1024 866 -> 566 us, 1024 x 4096 165 -> 121, 5120 x 256 120 -> 58, 256 x 1024 95 -> 32.
template <typename T, bool RAGGED>
__global__ void __launch_bounds__(512, 2) half_gemm_kernel(const HalfGemmArgs p) {
  __shared__ __align__(16) char lds[2 * kStage];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;

  // The first `whole` tiles are one workgroup's each, the others are dealt out in `splits` parts of their k's.
  const int tiles = ((p.M + kTile - 1) / kTile) * ((p.N + kTile - 1) / kTile), stages = (p.K + kBK - 1) / kBK;
  const bool is_part = (int)blockIdx.x >= p.whole;
  const int first = is_part ? p.whole : 0, count = is_part ? (tiles - p.whole) * p.splits : p.whole;
  int id = (int)blockIdx.x - first, part = 0, s_begin = 0, s_end = stages;
  const int xcd = id & 7, per = count >> 3, extra = count & 7;
  id = xcd * per + (xcd < extra ? xcd : extra) + (id >> 3);   // runs of neighbouring tiles for each XCD
  if (is_part) {
    part = id % p.splits;
    id = id / p.splits;
    s_begin = (int)((int64_t)stages * part / p.splits);
    s_end = (int)((int64_t)stages * (part + 1) / p.splits);
  }
  const Place at = place(p, first + id);

  float4v acc[8][4];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = float4v{0.0f, 0.0f, 0.0f, 0.0f};

  // This lane's 16 bytes of four k's of each operand's stage, 16 k's apart; columns past the end repeat the last ones.
  const int k_lane = wave * 2 + (lane >> 5);
  const int piece = (((lane >> 1) & 15) ^ order(k_lane)) * 2 + (lane & 1);   // (the same for all four)
  int am = piece * 8, bn = piece * 8;
  if (at.m0 + am > p.M - 8) am = p.M - 8 - at.m0;
  if (at.n0 + bn > p.N - 8) bn = p.N - 8 - at.n0;
  const uint32_t aoff = (uint32_t)(k_lane * (int)p.lda + at.m0 + am) * 2u, boff = (uint32_t)(k_lane * (int)p.ldb + at.n0 + bn) * 2u;
  const int64_t a_16 = 32 * p.lda, b_16 = 32 * p.ldb;   // bytes from one of the four to the next

  const int last = s_end > s_begin ? s_end - 1 : s_begin;   // past it, it is taken again, and never used
  const char *a, *b;
  int left;
  auto aim = [&](int s) {
    s = s < last ? s : last;
    a = (const char*)p.a + (int64_t)s * (4 * a_16);
    b = (const char*)p.b + (int64_t)s * (4 * b_16);
    left = p.K - s * kBK;
  };
  auto load = [&](const char* base, uint32_t off, char* dst, int i) {
    if (!RAGGED || left >= kBK) {
      const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(base), 0, 0xffffffffu, 0x00020000);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_ptr_t)dst, 16, off, 0, 0, 0);
    } else {   // the last stage: zeros past the last k
      uint4v v = {0u, 0u, 0u, 0u};
      if (i * 16 + k_lane < left) v = *(const __attribute__((address_space(1))) uint4v*)(base + off);
      *reinterpret_cast<uint4v*>(dst + lane * 16) = v;
    }
  };
  auto load_a = [&](int i, char* st) { load(a + i * a_16, aoff, st + i * 8192 + wave * 1024, i); };
  auto load_b = [&](int i, char* st) { load(b + i * b_16, boff, st + kPlane + i * 8192 + wave * 1024, i); };

  // Eight wavefronts of 128 x 64: eight and four operands of 16 columns, 32 k's at a time.
  const int wm = (wave >> 2) * 128, wn = (wave & 3) * 64;
  const int k_read = (lane >> 4) * 8 + ((lane & 15) >> 2);
  const int row_read = k_read * 512 + (lane & 3) * 8, ord = order(k_read);
  short8v af[2][4], bf[2][4];
  auto get_a = [&](const char* st, int half, int kh) {   // four of the eight
#pragma unroll
    for (int i = 0; i < 4; ++i) af[half][i] = read_across(st + kh * (32 * 512) + row_read + (((wm >> 4) + half * 4 + i) ^ ord) * 32);
  };
  auto get_b = [&](const char* st, int kh) {
#pragma unroll
    for (int j = 0; j < 4; ++j) bf[kh][j] = read_across(st + kPlane + kh * (32 * 512) + row_read + (((wn >> 4) + j) ^ ord) * 32);
  };
  auto product = [&](int i, int kh) {
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = mfma<T>(bf[kh][j], af[i >> 2][i & 3], acc[i][j]);
  };
  auto products = [&](int half, int kh) {
#pragma unroll
    for (int i = 0; i < 4; ++i) product(half * 4 + i, kh);
  };

  char* cur = lds;
  char* oth = lds + kStage;
  aim(s_begin);
#pragma unroll
  for (int i = 0; i < 4; ++i) { load_a(i, cur); load_b(i, cur); }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0), in a form the compiler's count of what is under way starts from
  asm volatile("s_barrier" ::: "memory");
  aim(s_begin + 1);
#pragma unroll
  for (int i = 0; i < 4; ++i) { load_a(i, oth); load_b(i, oth); }
  get_b(cur, 0);
  get_a(cur, 0, 0);
  for (int s = s_begin; s < s_end; ++s) {
    // Half of A's operands are multiplied while the next half is read.
    get_a(cur, 1, 0);
    __builtin_amdgcn_sched_barrier(0);
    products(0, 0);
    __builtin_amdgcn_sched_barrier(0);
    get_b(cur, 1);
    get_a(cur, 0, 1);
    __builtin_amdgcn_sched_barrier(0);
    products(1, 0);
    __builtin_amdgcn_sched_barrier(0);
    get_a(cur, 1, 1);
    __builtin_amdgcn_sched_barrier(0);
    products(0, 1);
    __builtin_amdgcn_sched_barrier(0);
    // All of this stage has been read, and all of the next one is there.
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    aim(s + 2);
    get_b(oth, 0);
    __builtin_amdgcn_sched_barrier(0);
    load_a(0, cur);
    load_b(0, cur);
    product(4, 1);
    __builtin_amdgcn_sched_barrier(0);
    get_a(oth, 0, 0);
    load_a(1, cur);
    load_b(1, cur);
    product(5, 1);
    __builtin_amdgcn_sched_barrier(0);
    load_a(2, cur);
    load_b(2, cur);
    product(6, 1);
    __builtin_amdgcn_sched_barrier(0);
    load_a(3, cur);
    load_b(3, cur);
    product(7, 1);
    __builtin_amdgcn_sched_barrier(0);
    char* x = cur;
    cur = oth;
    oth = x;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // no load into LDS outlives the workgroup

  // ---- store: a lane has four consecutive columns of one row of C ---------------------------------------------------
  const int r = wm + (lane & 15), c = wn + (lane >> 4) * 4;
  if (is_part) {
    float* dst = p.partial + ((int64_t)(at.tile - p.whole) * p.splits + part) * (kTile * kTile) + r * kTile + c;
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) *reinterpret_cast<float4v*>(dst + i * 16 * kTile + j * 16) = acc[i][j];
    return;
  }
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int row = at.m0 + r + i * 16, col = at.n0 + c + j * 16;
      if (row < p.M && col < p.N) {
        Words<T, 4> w;
        const float f[4] = {acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]};
        ElemBits<T>::template set<4>(w, f);
        *reinterpret_cast<uint2v*>((char*)p.c + ((int64_t)row * p.ldc + col) * 2) = uint2v{w.w[0], w.w[1]};
      }
    }
}

// The tiles that were dealt out in parts: their sum in a fixed order, eight columns per lane.
template <typename T>
__global__ void __launch_bounds__(256) half_reduce_kernel(const HalfGemmArgs p) {
  constexpr int kBlocks = kTile * kTile / 2048;   // per tile
  const Place to = place(p, p.whole + (int)blockIdx.x / kBlocks);
  const int at = ((int)blockIdx.x % kBlocks) * 2048 + (int)threadIdx.x * 8;
  const int row = to.m0 + at / kTile, col = to.n0 + at % kTile;
  if (row >= p.M || col >= p.N) return;
  const float* src = p.partial + (int64_t)(to.tile - p.whole) * p.splits * (kTile * kTile) + at;
  float4v lo = {0.0f, 0.0f, 0.0f, 0.0f}, hi = lo;
#pragma unroll 4
  for (int k = 0; k < p.splits; ++k) {
    lo += *reinterpret_cast<const float4v*>(src + (int64_t)k * (kTile * kTile));
    hi += *reinterpret_cast<const float4v*>(src + (int64_t)k * (kTile * kTile) + 4);
  }
  const float f[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  Words<T, 8> w;
  ElemBits<T>::template set<8>(w, f);
  *reinterpret_cast<uint4v*>((char*)p.c + ((int64_t)row * p.ldc + col) * 2) = uint4v{w.w[0], w.w[1], w.w[2], w.w[3]};
}

template <typename T>
void launch(const HalfGemmArgs& p, hipStream_t stream) {
  const int tiles = ((p.M + kTile - 1) / kTile) * ((p.N + kTile - 1) / kTile);
  const dim3 grid((unsigned)(p.whole + (tiles - p.whole) * p.splits));
  if (p.K % kBK != 0) hipLaunchKernelGGL((half_gemm_kernel<T, true>), grid, dim3(512), 0, stream, p);
  else hipLaunchKernelGGL((half_gemm_kernel<T, false>), grid, dim3(512), 0, stream, p);
  if (tiles > p.whole)
    hipLaunchKernelGGL(half_reduce_kernel<T>, dim3((unsigned)((tiles - p.whole) * (kTile * kTile / 2048))), dim3(256), 0, stream, p);
}

}  // namespace

void launch_half_gemm(int dtype, const HalfGemmArgs& p, hipStream_t stream) {
  if (dtype == QSSM_BF16) launch<bf16_t>(p, stream);
  else launch<f16_t>(p, stream);
}

}  // namespace qssm

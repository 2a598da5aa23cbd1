// Batched prefill kernels (gfx950): the decoder over all prompt tokens of
// several rows at once, M = tokens.  Same operations and rounding points as
// the decode step (batched_decoder_step.py:277-403), laid out for large M:
//
//   embed      token rows + per-token RoPE table
//   rmsnorm    one workgroup per token
//   GEMM       C[M,N] = A[M,K] W[N,K]^T, both operands K-contiguous.
//              bf16: MFMA v_mfma_f32_16x16x32_bf16, workgroup tiles of 256
//              (or 192) columns by 64 to 256 rows, K in steps of 64 through LDS
//              stages filled by direct global -> LDS loads, fp32
//              accumulation; epilogues "T(acc + bias)", the residual
//              "T(h + T(acc))", and gate/up with SwiGLU in one GEMM (the
//              tile's W rows half gate, half up); K split over workgroups
//              where the tiles alone leave CUs idle, the partial sums added
//              by the row kernel that follows.  fp32 models: 16 x 16 and
//              32 x 32 tiles on the fp32 MFMA, K split over a workgroup's
//              waves; 64 x 64 tiles through LDS on the vector units for large
//              products; the same epilogues.
//   qkv post   RoPE of q and k in place, K/V rows to their paged slots
//   attention  causal within each row's prompt.  bf16, head_dim 128: MFMA
//              for Q K^T and P V per (64-query tile, head), the softmax the
//              exact two-pass one of the decode step, the bf16 scores kept in
//              registers between the passes for prompts of up to 1,024 tokens
//              and computed again for longer ones; otherwise one workgroup
//              per (token, head).
#include <algorithm>
#include <type_traits>
#include <utility>

#include "re_device.h"
#include "re_layout.h"

namespace re {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef short lds_v4i16 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) lds_v4i16* lds_v4i16_ptr;
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

__device__ __forceinline__ bf16x8_t lds_frag(const bf16_t* p) {
  return __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const re_u32x4*>(p));
}

// ---------------------------------------------------------------------------
// Row kernels
// ---------------------------------------------------------------------------
// The partial sums of NV four-element vectors, added in range order; UNROLL
// ranges' loads in flight at once (each is a round trip to memory that
// another XCD wrote).  How many hardly matters: 2 to 14 at once with two vectors
// and 2 to 8 with four, four prompts of 2-5 tokens through 28 layers 3.31-3.33
// ms, of 37-250 tokens 9.69-9.75.
template <int NV, int UNROLL>
__device__ __forceinline__ void part_sums(const float* const (&p)[NV], size_t plane, int parts, re_f32x4 (&sum)[NV]) {
  int r = 0;
#pragma unroll
  for (int v = 0; v < NV; ++v) sum[v] = re_f32x4{0.f, 0.f, 0.f, 0.f};
  auto block = [&](auto n) {
    re_f32x4 x[n][NV];
#pragma unroll
    for (int u = 0; u < n; ++u)
#pragma unroll
      for (int v = 0; v < NV; ++v) x[u][v] = *reinterpret_cast<const re_f32x4*>(p[v] + (r + u) * plane);
#pragma unroll
    for (int u = 0; u < n; ++u)
#pragma unroll
      for (int v = 0; v < NV; ++v)
#pragma unroll
        for (int e = 0; e < 4; ++e) sum[v][e] += x[u][v][e];
    r += n;
  };
  while (r + UNROLL <= parts) block(std::integral_constant<int, UNROLL>{});
  while (r + 2 <= parts) block(std::integral_constant<int, 2>{});
  if (r < parts) block(std::integral_constant<int, 1>{});
}

template <typename T>
__global__ void __launch_bounds__(256) k_pf_embed(PrefillRows a) {
  const int m = blockIdx.x, tid = threadIdx.x;
  long long t = a.token[m];
  if (t < 0 || t >= a.V) t = 0;  // validated on the host; reads stay in bounds
  const int half = a.head_dim / 2;
  for (int j = tid; j < half; j += blockDim.x) {
    const float ang = static_cast<float>(a.pos[m]) * a.inv_freq[j];
    a.rope[((size_t)m * half + j) * 2] = Elt<T>::r(cosf(ang));
    a.rope[((size_t)m * half + j) * 2 + 1] = Elt<T>::r(sinf(ang));
  }
  const T* src = static_cast<const T*>(a.embedding) + (size_t)t * a.H;
  T* dst = static_cast<T*>(a.hidden) + (size_t)m * a.H;
  for (int c = tid; c < a.H / 8; c += blockDim.x)
    *reinterpret_cast<Vec8<T>*>(dst + c * 8) = Vec8<T>::load_cached(src + c * 8);
}

// RMSNorm (batched_decoder_step.py:224-229): fp32 mean of squares, rsqrt,
// cast to T, T x T product with the weight.  One workgroup per token, its row
// in registers (H <= 4,096).
//
// PART: the residual add of the preceding split GEMM comes first, h =
// T(h + T(p_0 + p_1 + ...)) over its fp32 partials [parts][M][H] in range
// order (the residual epilogue's roundings), written back to x.
// PART runs one 8-element vector per thread (512 threads), so all of a row's
// partials are on their way in two or three round trips.
constexpr int kNormRow = 4096;
template <typename T, bool PART>
__global__ void __launch_bounds__(PART ? 512 : 256) k_pf_rmsnorm(void* x, const void* w, void* y, int H, float eps,
                                                                 const float* part, int parts) {
  constexpr int kThreads = PART ? 512 : 256, kNormVecs = kNormRow / 8 / kThreads;
  __shared__ float red[kThreads / 64];
  const int m = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  T* xr = static_cast<T*>(x) + (size_t)m * H;
  const T* wr = static_cast<const T*>(w);
  T* yr = static_cast<T*>(y) + (size_t)m * H;
  const size_t plane = (size_t)gridDim.x * H;
  Vec8<T> v[kNormVecs];
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < kNormVecs; ++i) {
    const int c = tid + kThreads * i;
    if (c * 8 >= H) continue;
    v[i] = Vec8<T>::load_cached(xr + c * 8);
    if constexpr (PART) {
      const float* p0 = part + (size_t)m * H + c * 8;
      const float* const p[2] = {p0, p0 + 4};
      re_f32x4 ps[2];
      part_sums<2, 7>(p, plane, parts, ps);
      float nh[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) nh[e] = Elt<T>::r(v[i].get(e) + Elt<T>::r(ps[e >> 2][e & 3]));
      v[i] = Vec8<T>::from_floats(nh);
      *reinterpret_cast<Vec8<T>*>(xr + c * 8) = v[i];
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) s = fmaf(v[i].get(e), v[i].get(e), s);
  }
  s = wave_sum(s);
  if (lane == 0) red[wave] = s;
  __syncthreads();
  float total = red[0];
#pragma unroll
  for (int i = 1; i < kThreads / 64; ++i) total += red[i];
  const float rs = rsqrtf(total / static_cast<float>(H) + eps);
#pragma unroll
  for (int i = 0; i < kNormVecs; ++i) {
    const int c = tid + kThreads * i;
    if (c * 8 >= H) continue;
    const Vec8<T> g = Vec8<T>::load_cached(wr + c * 8);
    float out[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) out[e] = Elt<T>::r(Elt<T>::r(v[i].get(e) * rs) * g.get(e));
    *reinterpret_cast<Vec8<T>*>(yr + c * 8) = Vec8<T>::from_floats(out);
  }
}

// RoPE of q and k (rows already rounded with their bias) in place, and the
// paged slot write of k and v (batched_decoder_step.py:231-264, 323-324).
template <typename T>
__device__ __forceinline__ void store8(T* p, const Vec8<T>& v);
template <>
__device__ __forceinline__ void store8<bf16_t>(bf16_t* p, const Vec8<bf16_t>& v) {
  *reinterpret_cast<re_u32x4*>(p) = v.v;
}
template <>
__device__ __forceinline__ void store8<float>(float* p, const Vec8<float>& v) {
  reinterpret_cast<re_f32x4*>(p)[0] = v.a;
  reinterpret_cast<re_f32x4*>(p)[1] = v.b;
}

// One workgroup per token; a thread takes 8 consecutive pair indices j of one
// head (16-byte accesses of both halves, the RoPE table's 8 cos/sin pairs),
// head_dim a multiple of 16.
//
// PART: the rows come from the split GEMM's fp32 partials instead, T(p_0 +
// p_1 + ... + bias) (the store epilogue's rounding), v written to the rows too.
// Its workgroups have a thread per vector pair where 512 threads allow it.
template <typename T, bool PART>
__global__ void __launch_bounds__(PART ? 512 : 256) k_pf_qkv_post(PrefillQkv a) {
  const int m = blockIdx.x;
  const int half = a.head_dim / 2, hv = half / 8;
  const int nq = a.heads, nkv = a.kv_heads;
  T* row = static_cast<T*>(a.qkv) + (size_t)m * a.ld;
  const int s = a.slot[m];
  const bool to_cache = s >= 0 && s < a.slots;
  const float* rope = a.rope + (size_t)m * half * 2;
  for (int idx = threadIdx.x; idx < (nq + 2 * nkv) * hv; idx += blockDim.x) {
    const int hg = idx / hv, j = (idx - hg * hv) * 8;
    T* p = row + (size_t)hg * a.head_dim;
    Vec8<T> va, vb;
    if constexpr (PART) {
      const int n0 = hg * a.head_dim + j, np = (nq + 2 * nkv) * a.head_dim;
      const float* pp = a.part + (size_t)m * np + n0;
      const float* const ps[4] = {pp, pp + 4, pp + half, pp + half + 4};
      re_f32x4 sum[4];
      part_sums<4, 5>(ps, (size_t)a.M * np, a.parts, sum);
      float sa[8], sb[8];
      const T* bias = static_cast<const T*>(a.bias) + n0;
      const Vec8<T> ba = Vec8<T>::load_cached(bias), bb = Vec8<T>::load_cached(bias + half);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        sa[e] = Elt<T>::r(sum[e >> 2][e & 3] + ba.get(e));
        sb[e] = Elt<T>::r(sum[2 + (e >> 2)][e & 3] + bb.get(e));
      }
      va = Vec8<T>::from_floats(sa);
      vb = Vec8<T>::from_floats(sb);
    } else {
      va = Vec8<T>::load_cached(p + j);
      vb = Vec8<T>::load_cached(p + j + half);
    }
    if (hg < nq + nkv) {
      float oa[8], ob[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float c = rope[(j + e) * 2], sn = rope[(j + e) * 2 + 1];
        const float qa = va.get(e), qb = vb.get(e);
        oa[e] = Elt<T>::r(Elt<T>::r(qa * c) + Elt<T>::r(-qb * sn));
        ob[e] = Elt<T>::r(Elt<T>::r(qb * c) + Elt<T>::r(qa * sn));
      }
      va = Vec8<T>::from_floats(oa);
      vb = Vec8<T>::from_floats(ob);
    }
    if (PART || hg < nq + nkv) {
      store8<T>(p + j, va);
      store8<T>(p + j + half, vb);
    }
    if (hg >= nq && to_cache) {
      const bool is_key = hg < nq + nkv;
      const int kvh = is_key ? hg - nq : hg - nq - nkv;
      T* cache = static_cast<T*>(is_key ? a.key_cache : a.value_cache) + ((size_t)s * nkv + kvh) * a.head_dim;
      store8<T>(cache + j, va);
      store8<T>(cache + j + half, vb);
    }
  }
}

// ---------------------------------------------------------------------------
// GEMMs
// ---------------------------------------------------------------------------
// bf16: one 64 MJ x 256 output tile (MJ = 1 .. 4) per workgroup of 8 waves, K
// in steps of 64, over all of K or over one of nS ranges of it.
//
// Operands reach LDS by direct global -> LDS loads (global_load_lds_dwordx4,
// 16 bytes per lane, no register staging) into ST stages of 32 + 8 MJ KB: W
// tile rows 0..255, then the A tile's rows, 128 bytes (one K step) per row.
// Chunk c (16 bytes) of row r sits in slot c ^ gemm_swz(r), so the fragment
// reads below hit distinct banks for 8 and for 16 consecutive rows.  The
// products run as C^T = W A^T on v_mfma_f32_16x16x32_bf16: wave (wn, wm) owns
// NI x MI tiles of 16 x 16 (n x m, gemm_waves_n), and a lane's accumulator holds
// four consecutive output columns of one row.  A stage is two sub-steps of K =
// 32; each sub-step's NI + MI fragments are read under the previous sub-step's
// NI MI products.  The stage's one barrier sits between its sub-steps: before it
// each wave waits for its own loads of stage kt + 1 and its reads of stage
// kt, so after it stage kt + 1 is complete in LDS and stage kt's buffer is
// free.  The loads of stage kt + ST go out during the second sub-step (waves
// 0-3 at its start, waves 4-7 after 3/8 of their products, so the two waves
// of a SIMD do not stall on them together), and stage kt + 1's first
// fragments are read under the second sub-step's products, so no wave waits
// on LDS at a stage boundary.  The epilogue rounds the tile to bf16 in LDS
// (rows padded to 264 elements) and writes it as row-contiguous 16-byte
// vectors: "T(acc + bias)" (qkv), or the residual "T(h + T(acc))"; a K range's
// sums leave as fp32 from the accumulators, for the next launch to add.
//
// What bounds it: 256-row tiles the loop that feeds the matrix cores from LDS
// (about 1.2 us a stage with every CU busy, 0.5 of the bf16 peak).  A call of
// few rows has few tiles (14-18 for the 3,584- and 4,608-column products of
// up to 256 rows on 256 CUs) and is bound by that serial loop, not by memory;
// lower tiles shorten a stage (0.66 us at 64 rows, where three stages fit LDS
// and 80 KB of loads stay in flight), K ranges the number of stages.
//
// Workgroups are dispatched round-robin over the 8 XCDs; workgroup b runs
// tile t = (b % 8) * ceil(T / 8) + b / 8 of an order with the K ranges
// outermost and the tiles of a range grouped (4 M tiles by every N tile), so
// the 32 tiles an XCD runs at once share 4 A and 8 W row blocks in its L2,
// and the tiles of a K range share its columns of A.  Up to 8 M tiles are one
// group, so W is read through once (gate/up at 400 tokens, 64-row tiles: 210
// -> 186 us in one group of 7 instead of groups of 4 and 3; at 570 and 1,000
// tokens, 128-row tiles, 171.6 -> 169.7 and 281.8 -> 278.0).
//
// Requirements (checked by launch_gemm): K % 64 == 0, N % 8 == 0, lda, ldw
// and ldo multiples of 8 elements, 16-byte aligned operands.
constexpr int kGn = 256, kGk = 64;
constexpr int kGnNarrow = 192;
constexpr int kGrowBytes = kGk * 2;                   // one K step of one row
constexpr int kGwaves = 8, kGthreads = kGwaves * 64;
constexpr int kGgroupM = 4;
constexpr int gemm_tile_m(int mj) { return 64 * mj; }
constexpr int gemm_stage_bytes(int mj, int gn) { return (gn + gemm_tile_m(mj)) * kGrowBytes; }
constexpr int gemm_stages(int mj) { return mj <= 2 ? 3 : 2; }
constexpr int gemm_out_ld(int gn) { return gn + 8; }  // epilogue row stride (elements)
constexpr int gemm_lds_bytes(int mj, int st, int gn) {
  return std::max(gemm_tile_m(mj) * gemm_out_ld(gn) * 2, st * gemm_stage_bytes(mj, gn));
}

typedef const __attribute__((address_space(1))) void* gemm_gptr;
typedef __attribute__((address_space(3))) void* gemm_lptr;

__device__ __forceinline__ int gemm_swz(int r) { return (r & 7) ^ ((r >> 3) & 1); }

// s_waitcnt immediate: vmcnt <= vm (6 bits), lgkmcnt 0, expcnt untouched.
constexpr int gemm_wait_vm(int vm) { return (vm & 15) | ((vm >> 4) << 14) | (7 << 4); }

// End of a stage: this wave's LDS reads and all but the last VM of its loads
// are done, then the barrier.  The empty asm statements keep the compiler
// from moving memory accesses across; the wait is a real instruction the
// wait-count pass accounts for.
template <int VM = 0>
__device__ __forceinline__ void gemm_stage_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(gemm_wait_vm(VM));
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("" ::: "memory");
}

// Tile and K range of workgroup b (see above): K ranges outermost.
__device__ __forceinline__ void gemm_tile_of(int b, int nM, int nN, int nS, int& mt, int& nt, int& ks) {
  const int tiles = nM * nN, total = tiles * nS, x = b & 7, local = b >> 3, q = total >> 3, r = total & 7;
  int t = x < r ? x * (q + 1) + local : r * (q + 1) + (x - r) * q + local;
  ks = t / tiles;
  t -= ks * tiles;
  const int group_m = nM <= 2 * kGgroupM ? nM : kGgroupM;
  const int per_group = group_m * nN, g = t / per_group, first = g * group_m;
  const int gm = min(group_m, nM - first), w = t - g * per_group;
  mt = first + w % gm;
  nt = w / gm;
}

// Waves along n: a wave's block of 16 x 16 tiles is 8 x 4 (n x m) of a 256-row
// tile and 4 x 6, 4 x 4 and 4 x 2 of the lower ones, the fewest fragment reads
// per product (two waves along n throughout: 11 reads for 24 products, 10 for
// 16 and 9 for 8 instead of 10, 8 and 6).  Gate/up at 570 tokens, 128-row tiles:
// 181 -> 171 us; 400 tokens 170 -> 161; 2,000 tokens, 64-row tiles 811 -> 774;
// 192-row tiles the same within 1 %.
constexpr int gemm_waves_n(int mj) { return mj == 4 ? 2 : 4; }

// Fragments of the next stage read before product p of the second sub-step:
// one per two products where that covers them, else spread over the first 7/8
// of the products.
constexpr int gemm_reads_by(int frags, int prods, int p) {
  const int span = prods - prods / 8;
  const int n = 2 * frags <= prods ? p / 2 : (p * frags + span - 1) / span;
  return n < frags ? n : frags;
}

template <int EPI, int MJ, int ST, int GN>
__global__ void __launch_bounds__(kGthreads, 1) k_gemm_bf16(GemmArgs a, int nM, int nN, int nS) {
  extern __shared__ __align__(16) unsigned char gsm[];
  constexpr int kTm = gemm_tile_m(MJ), kStage = gemm_stage_bytes(MJ, GN), kOutLd = gemm_out_ld(GN);
  constexpr int kWInsts = GN / 64, kInsts = kWInsts + MJ;  // 1 KB loads (8 rows) of each wave and stage
  // wave-uniform, so the load base lives in SGPRs (32-bit per-lane offsets)
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_index(tid);
  int mt, nt, ks;
  gemm_tile_of(blockIdx.x, nM, nN, nS, mt, nt, ks);
  // The SwiGLU tile covers GN / 2 output columns: the first half of the W tile
  // rows are their gate rows, the second half their up rows.
  constexpr bool kPart = EPI == kGemmPart;
  constexpr bool kSwiGlu = EPI == kGemmSwiGlu;
  constexpr int kTileN = kSwiGlu ? GN / 2 : GN;
  const int m0 = mt * kTm, n0 = nt * kTileN;
  // K steps of this workgroup: range ks of nS nearly equal ones
  const int steps = a.K / kGk;
  const int k_begin = kPart ? static_cast<int>((long long)ks * steps / nS) : 0;
  const int nk = (kPart ? static_cast<int>((long long)(ks + 1) * steps / nS) : steps) - k_begin;
  // Loads.  256-row tiles: waves 0-3 bring W rows 0..255, waves 4-7 A rows
  // 0..255.  Smaller ones: every wave GN / 8 W rows (4 loads of 8, or 3 of the
  // 192-wide tile) and 8 MJ A rows.
  // Rows past M or N read a valid row (clamped) whose results are never stored.
  constexpr bool kSplitLoads = MJ == 4;
  static_assert(!kSplitLoads || GN == kGn, "256-row tiles are 256 wide");
  const char* wbase;
  const char* abase = static_cast<const char*>(a.A) + (size_t)m0 * a.lda * 2 + (size_t)k_begin * kGrowBytes;
  uint32_t goff[kInsts];
  int lrow[2];  // tile row of the wave's first W (or only) load and of its first A load
  if constexpr (kSplitLoads) {
    const int row0 = wave * 64;
    const bool loads_w = row0 < kGn;
    const void* wsrc = kSwiGlu && row0 >= kTileN ? a.W2 : a.W;
    wbase = loads_w ? static_cast<const char*>(wsrc) + (size_t)n0 * a.ldw * 2 + (size_t)k_begin * kGrowBytes : abase;
    const long long ld = loads_w ? a.ldw : a.lda;
    const int rows_left = loads_w ? a.N - n0 : a.M - m0;
#pragma unroll
    for (int i = 0; i < kInsts; ++i) {
      // lane l of instruction i writes slot l % 8 of row row0 + 8 i + l / 8
      const int row = row0 + i * 8 + (lane >> 3);
      const int chunk = (lane & 7) ^ gemm_swz(row);
      const int local = loads_w ? row % kTileN : row & 255;  // the row within its source matrix
      goff[i] = static_cast<uint32_t>(min(local, rows_left - 1) * ld * 2 + chunk * 16);
    }
    lrow[0] = lrow[1] = row0;
  } else {
    lrow[0] = wave * (GN / 8);
    lrow[1] = GN + wave * 8 * MJ;
    const void* wsrc = kSwiGlu && lrow[0] >= kTileN ? a.W2 : a.W;
    wbase = static_cast<const char*>(wsrc) + (size_t)n0 * a.ldw * 2 + (size_t)k_begin * kGrowBytes;
#pragma unroll
    for (int i = 0; i < kInsts; ++i) {
      const int row = (i < kWInsts ? lrow[0] + i * 8 : lrow[1] + (i - kWInsts) * 8) + (lane >> 3);
      const int chunk = (lane & 7) ^ gemm_swz(row);
      goff[i] = i < kWInsts ? static_cast<uint32_t>(min(row % kTileN, a.N - n0 - 1) * a.ldw * 2 + chunk * 16)
                      : static_cast<uint32_t>(min(row - GN, a.M - m0 - 1) * a.lda * 2 + chunk * 16);
    }
  }
  auto issue = [&](int kt, int buf) {
    const size_t kb = (size_t)kt * kGrowBytes;
    unsigned char* l = gsm + buf * kStage;
    if constexpr (kSplitLoads) {
#pragma unroll
      for (int i = 0; i < kInsts; ++i)
        __builtin_amdgcn_global_load_lds((gemm_gptr)(wbase + kb + goff[i]),
                                         (gemm_lptr)(l + lrow[0] * kGrowBytes + i * 1024), 16, 0, 0);
    } else {
#pragma unroll
      for (int i = 0; i < kWInsts; ++i)
        __builtin_amdgcn_global_load_lds((gemm_gptr)(wbase + kb + goff[i]),
                                         (gemm_lptr)(l + lrow[0] * kGrowBytes + i * 1024), 16, 0, 0);
#pragma unroll
      for (int i = kWInsts; i < kInsts; ++i)
        __builtin_amdgcn_global_load_lds((gemm_gptr)(abase + kb + goff[i]),
                                         (gemm_lptr)(l + lrow[1] * kGrowBytes + (i - kWInsts) * 1024), 16, 0, 0);
    }
  };
  constexpr int kWn = gemm_waves_n(MJ), NI = GN / 16 / kWn, MI = 4 * MJ / (kGwaves / kWn);
  const int wn = wave % kWn, wm = wave / kWn;
  f32x4_t acc[NI][MI];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < MI; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) acc[i][j][v] = 0.f;
  // lane l supplies row l % 16 of a 16-row operand tile, K elements
  // 8 (l / 16) ..+8 of the 32-wide sub-step
  const int fr = lane & 15, fq = lane >> 4;
  // (16-row tiles start at multiples of 16, so their row's swizzle is fr's)
  const int frag_off[2] = {fr * kGrowBytes + ((fq ^ gemm_swz(fr)) * 16), fr * kGrowBytes + (((4 + fq) ^ gemm_swz(fr)) * 16)};
  auto frag = [&](int st, int row0, int ks2) -> bf16x8_t {
    return lds_frag(reinterpret_cast<const bf16_t*>(gsm + st * kStage + row0 * kGrowBytes + frag_off[ks2]));
  };
  // First W tile row of the wave's block i.  kGlu: blocks 0 .. NI / 2 - 1 are
  // gate rows and the rest the up rows of the same columns, so a lane holds
  // both of an output and half as much goes through LDS in the epilogue (32,000
  // tokens 7,140 -> 7,036 us, 570 tokens in 192-row tiles 181 -> 177).  The
  // 192-wide tiles have three blocks per wave and pair them up in LDS.
  constexpr bool kGlu = kSwiGlu && NI % 2 == 0;
  constexpr int kHalfNI = NI / 2;
  auto w_block = [&](int i) {
    if constexpr (kGlu) return (wn * kHalfNI + i % kHalfNI) * 16 + (i < kHalfNI ? 0 : kTileN);
    return (wn * NI + i) * 16;
  };
  // fragment sets: [set][0 .. NI - 1] W rows (n), [set][NI ..] A rows (m)
  constexpr int kFrags = NI + MI, kProds = NI * MI;
  bf16x8_t f[2][kFrags];
  auto read_frag = [&](int set, int idx, int st, int ks2) {
    f[set][idx] = idx < NI ? frag(st, w_block(idx), ks2) : frag(st, GN + (wm * MI + idx - NI) * 16, ks2);
  };
  auto read_set = [&](int set, int st, int ks2) {
#pragma unroll
    for (int i = 0; i < kFrags; ++i) read_frag(set, i, st, ks2);
  };
  auto products = [&](int set) {
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int j = 0; j < MI; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[set][i], f[set][NI + j], acc[i][j], 0, 0, 0);
#pragma unroll
    for (int r = 0; r < kFrags; ++r) {  // fragment reads spread over the products
      __builtin_amdgcn_sched_group_barrier(0x008, kProds / kFrags > 0 ? kProds / kFrags : 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // Stages 0..ST-1 go out at once.  With 256-row tiles and one K range a
  // stage past the end re-reads the last one (never used): without the branch
  // around the loads the loop is 0.6 % faster, and K is long.  Elsewhere
  // (ranges of a few stages) a stage that does not exist is not read.
  constexpr bool kAlways = MJ == 4 && !kPart;
  const int first = kAlways ? ST : min(ST, nk);
  for (int s = 0; s < first; ++s) issue(kAlways ? min(s, nk - 1) : s, s);
  if (first == ST)
    __builtin_amdgcn_s_waitcnt(gemm_wait_vm((ST - 1) * kInsts));  // this wave's stage 0
  else
    __builtin_amdgcn_s_waitcnt(gemm_wait_vm(0));
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  read_set(0, 0, 0);
  __builtin_amdgcn_sched_barrier(0);
  int ring = 0;
  for (int kt = 0; kt < nk; ++kt) {
    const int st = ST == 2 ? kt & 1 : ring, nst = ST == 2 ? st ^ 1 : ring + 1 == ST ? 0 : ring + 1;
    read_set(1, st, 1);
    products(0);
    // stage kt + 1 complete (stages kt + 2 .. kt + ST - 1 may be in flight),
    // stage kt's buffer free
    if (ST > 2 && kt + ST - 1 < nk)
      gemm_stage_barrier<(ST - 2) * kInsts>();
    else
      gemm_stage_barrier();
    const bool more = kAlways || kt + ST < nk;
    const int next = kAlways ? min(kt + ST, nk - 1) : kt + ST;
    // Second sub-step, in a fixed order: the products row block by row block,
    // the next stage's first fragments between them (past the last stage: a
    // stale buffer, never used), and the loads of stage kt + ST.  The two
    // waves of a SIMD (w and w + 4) issue their loads apart: an issuing wave
    // waits while the memory pipeline takes its 1 KB requests, and meanwhile
    // the other wave's products run.
#pragma unroll
    for (int p = 0; p < kProds; ++p) {
      const int i = p / MI, j = p % MI;
      if (p == 0 && wave < 4 && more) issue(next, st);
      if (p == kProds * 3 / 8 && wave >= 4 && more) issue(next, st);
      if (j == 0) __builtin_amdgcn_sched_barrier(0);
      acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[1][i], f[1][NI + j], acc[i][j], 0, 0, 0);
#pragma unroll
      for (int r = gemm_reads_by(kFrags, kProds, p); r < gemm_reads_by(kFrags, kProds, p + 1); ++r) read_frag(0, r, nst, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    ring = nst;
  }
  // acc[i][j] value v of lane l: n = 16 i + 4 (l / 16) + v, m = 16 j + l % 16
  // within the wave's block
  if constexpr (kPart) {
    // fp32 partial sums [nS][M][N], four consecutive columns per lane
#pragma unroll
    for (int j = 0; j < MI; ++j)
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int m = m0 + (wm * MI + j) * 16 + fr, n = n0 + (wn * NI + i) * 16 + 4 * fq;
        if (m < a.M && n < a.N)
          *reinterpret_cast<f32x4_t*>(a.part + ((size_t)ks * a.M + m) * a.N + n) = acc[i][j];
      }
    return;
  }
  gemm_stage_barrier();
  bf16_t* T = reinterpret_cast<bf16_t*>(gsm);
  if constexpr (kGlu) {
    // silu as the decode step computes it, rounded, then the rounded product
    constexpr int kLd = gemm_out_ld(kTileN);
#pragma unroll
    for (int j = 0; j < MI; ++j)
#pragma unroll
      for (int i = 0; i < kHalfNI; ++i) {
        const int ml = (wm * MI + j) * 16 + fr, nl = (wn * kHalfNI + i) * 16 + 4 * fq;
        float y[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float x = round_bf16(acc[i][j][e]);
          y[e] = round_bf16(x / (1.0f + expf(-x))) * round_bf16(acc[i + kHalfNI][j][e]);
        }
        *reinterpret_cast<uint2*>(T + ml * kLd + nl) = make_uint2(f2_to_bf16x2(y[0], y[1]), f2_to_bf16x2(y[2], y[3]));
      }
    gemm_stage_barrier();
    bf16_t* out = static_cast<bf16_t*>(a.out);
#pragma unroll 4
    for (int idx = tid; idx < kTm * kTileN / 8; idx += kGthreads) {
      const int r = idx / (kTileN / 8), c = idx % (kTileN / 8);
      const int m = m0 + r, n = n0 + c * 8;
      if (m < a.M && n < a.N)
        *reinterpret_cast<re_u32x4*>(out + (size_t)m * a.ldo + n) = *reinterpret_cast<const re_u32x4*>(T + r * kLd + c * 8);
    }
    return;
  }
  const bf16_t* bias = static_cast<const bf16_t*>(a.bias);
#pragma unroll
  for (int j = 0; j < MI; ++j)
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int ml = (wm * MI + j) * 16 + fr, nl = (wn * NI + i) * 16 + 4 * fq;
      float y[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = acc[i][j][e];
      if (EPI == kGemmStore && bias != nullptr) {
        const uint2 b = *reinterpret_cast<const uint2*>(bias + min(n0 + nl, a.N - 4));
        y[0] += __uint_as_float(b.x << 16);
        y[1] += __uint_as_float(b.x & 0xffff0000u);
        y[2] += __uint_as_float(b.y << 16);
        y[3] += __uint_as_float(b.y & 0xffff0000u);
      }
      *reinterpret_cast<uint2*>(T + ml * kOutLd + nl) =
          make_uint2(f_to_bf16(y[0]) | ((uint32_t)f_to_bf16(y[1]) << 16),
                     f_to_bf16(y[2]) | ((uint32_t)f_to_bf16(y[3]) << 16));
    }
  gemm_stage_barrier();
  bf16_t* out = static_cast<bf16_t*>(a.out);
  if constexpr (kSwiGlu) {
    // columns c of the gate half and 128 + c of the up half give output
    // column n0 + c: silu as the decode step computes it, rounded, then the
    // rounded product
#pragma unroll 4
    for (int idx = tid; idx < kTm * kTileN / 8; idx += kGthreads) {
      const int r = idx / (kTileN / 8), c = idx % (kTileN / 8);
      const int m = m0 + r, n = n0 + c * 8;
      if (m >= a.M || n >= a.N) continue;
      const Vec8<bf16_t> gv = Vec8<bf16_t>::load_cached(T + r * kOutLd + c * 8);
      const Vec8<bf16_t> uv = Vec8<bf16_t>::load_cached(T + r * kOutLd + kTileN + c * 8);
      float y[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float x = gv.get(e);
        const float sg = round_bf16(x / (1.0f + expf(-x)));
        y[e] = round_bf16(sg * uv.get(e));
      }
      *reinterpret_cast<Vec8<bf16_t>*>(out + (size_t)m * a.ldo + n) = Vec8<bf16_t>::from_floats(y);
    }
    return;
  }
#pragma unroll 4
  for (int idx = tid; idx < kTm * GN / 8; idx += kGthreads) {
    const int r = idx / (GN / 8), c = idx % (GN / 8);
    const int m = m0 + r, n = n0 + c * 8;
    if (m >= a.M || n >= a.N) continue;
    re_u32x4 t = *reinterpret_cast<const re_u32x4*>(T + r * kOutLd + c * 8);
    re_u32x4* p = reinterpret_cast<re_u32x4*>(out + (size_t)m * a.ldo + n);
    if constexpr (EPI == kGemmResidual) {
      const re_u32x4 h = *p;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float lo = __uint_as_float(h[e] << 16) + __uint_as_float(t[e] << 16);
        const float hi = __uint_as_float(h[e] & 0xffff0000u) + __uint_as_float(t[e] & 0xffff0000u);
        t[e] = f_to_bf16(lo) | ((uint32_t)f_to_bf16(hi) << 16);
      }
    }
    *p = t;
  }
}

// fp32 models, large products: 64 x 64 tiles through LDS on the vector units, 4
// x 4 sums per thread, K in steps of 16.  SwiGLU: 32 output columns, in LDS two
// gate rows and their two up rows in turn, so a thread's four sums of a row are
// gate and up of two columns and the launch has as many workgroups as the two
// products.  Bound by the vector units' rate and LDS reads, 70-77 TFLOP/s;
// the matrix-core kernel below reads its operands from L2 for every 32 x 32 tile
// and stays at 60 (22-27 where it has to load element by element).  See
// gemm_f32_launch.  Eight workgroups per CU (64 registers): at seven, 3,424 x
// 2,235 x 1,348 takes 352 us instead of 333.  m_on_x: the grid's first dimension
// runs over M tiles, else over N tiles.
template <int EPI>
__global__ void __launch_bounds__(256, 8) k_gemm_f32_lds(GemmArgs a, int m_on_x) {
  constexpr bool kSwiGlu = EPI == kGemmSwiGlu;
  constexpr int kTileN = kSwiGlu ? 32 : 64;
  __shared__ float As[16][64 + 4];
  __shared__ float Ws[16][64 + 4];
  const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
  const int m0 = (m_on_x ? blockIdx.x : blockIdx.y) * 64, n0 = (m_on_x ? blockIdx.y : blockIdx.x) * kTileN;
  const float* A = static_cast<const float*>(a.A);
  float acc[4][4] = {};
  for (int k0 = 0; k0 < a.K; k0 += 16) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      // rows past M or N read a valid row (clamped) whose results are never stored
      const int idx = tid + 256 * i, row = idx >> 4, kk = idx & 15, k = k0 + kk;
      const bool kin = k < a.K;
      const float* W = static_cast<const float*>(kSwiGlu && i >= 2 ? a.W2 : a.W);  // rows 32.. from i = 2 on
      const float x = A[(size_t)min(m0 + row, a.M - 1) * a.lda + (kin ? k : 0)];
      const float y = W[(size_t)min(n0 + row % kTileN, a.N - 1) * a.ldw + (kin ? k : 0)];
      As[kk][row] = kin ? x : 0.f;
      Ws[kk][kSwiGlu ? (row % 32 / 2) * 4 + (row / 32) * 2 + row % 2 : row] = kin ? y : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < 16; ++kk) {
      float av[4], wv[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        av[r] = As[kk][ty * 4 + r];
        wv[r] = Ws[kk][tx * 4 + r];
      }
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[r][c] = fmaf(av[r], wv[c], acc[r][c]);
    }
    __syncthreads();
  }
  float* out = static_cast<float*>(a.out);
  const float* bias = static_cast<const float*>(a.bias);
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int c = 0; c < (kSwiGlu ? 2 : 4); ++c) {
      const int m = m0 + ty * 4 + r, n = n0 + tx * (kSwiGlu ? 2 : 4) + c;
      if (m >= a.M || n >= a.N) continue;
      float* o = out + (size_t)m * a.ldo + n;
      const float y = acc[r][c];
      if constexpr (EPI == kGemmStore)
        *o = y + (bias != nullptr ? bias[n] : 0.f);
      else if constexpr (EPI == kGemmResidual)
        *o = *o + y;
      else
        *o = y / (1.0f + expf(-y)) * acc[r][c + 2];
    }
}

// fp32 models, smaller products: one 16 MT x 16 MT output tile per workgroup of
// four waves, on
// v_mfma_f32_16x16x4_f32 (fp32 operands and sums).  K goes to the waves in
// 16-element chunks, chunk c to wave c % 4, so the workgroup reads its rows in
// contiguous 256-byte pieces; a lane takes four consecutive K elements of its
// row of each operand straight from memory (16 bytes), and instruction e of a
// chunk multiplies element e of every lane: its four k indexes are elements
// e, 4 + e, 8 + e and 12 + e of the chunk, in both operands alike.  As in the
// bf16 kernel the products run as C^T = W A^T.  The four waves' sums are added
// in wave order through LDS.  K need not be a multiple of anything and the
// operands need no alignment past 4 bytes: VEC = false loads element by
// element.
//
// What bounds it: the products are small (the tiny test model: 66 tokens,
// K = 256 and 688), so latency does: one chain of loads per K chunk.  The
// chunks are spread over four waves and UN of them are in flight at once, and
// the tile is 16 x 16 while 32 x 32 would not give every CU two workgroups.
// 66 tokens, before (64 x 64 tiles through LDS on the vector units) and now:
// K = 256, N = 512 24.2 -> 3.8 us; K = 688, N = 256 63.7 -> 5.0 us.
//
// SwiGLU: W the gate rows, W2 the up rows, out = silu(gate) * up.
template <int EPI, int MT, bool VEC>
__global__ void __launch_bounds__(256) k_gemm_f32(GemmArgs a, int nN) {
  constexpr int kT = 16 * MT, kOps = EPI == kGemmSwiGlu ? 2 : 1, kLd = kT + 4;
  constexpr int UN = MT == 1 ? 4 : 2;
  __shared__ __align__(16) float red[4][kOps][kT][kLd];
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_index(tid);
  const int m0 = blockIdx.x / nN * kT, n0 = blockIdx.x % nN * kT;
  const int fr = lane & 15, fq = lane >> 4;
  // Rows past M or N read a valid row (clamped) whose results are never stored.
  const float* arow[MT];
  const float* wrow[kOps][MT];
#pragma unroll
  for (int j = 0; j < MT; ++j) {
    arow[j] = static_cast<const float*>(a.A) + (size_t)min(m0 + 16 * j + fr, a.M - 1) * a.lda;
#pragma unroll
    for (int b = 0; b < kOps; ++b)
      wrow[b][j] = static_cast<const float*>(b == 0 ? a.W : a.W2) + (size_t)min(n0 + 16 * j + fr, a.N - 1) * a.ldw;
  }
  // four elements of a row from k on; zero past K
  auto load4 = [&](const float* row, int k) -> f32x4_t {
    f32x4_t v = {0.f, 0.f, 0.f, 0.f};
    if constexpr (VEC) {
      if (k < a.K) v = *reinterpret_cast<const f32x4_t*>(row + k);  // K % 4 == 0
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (k + e < a.K) v[e] = row[k + e];
    }
    return v;
  };
  f32x4_t acc[kOps][MT][MT];  // [operand][n][m]
#pragma unroll
  for (int b = 0; b < kOps; ++b)
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < MT; ++j) acc[b][i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  for (int k0 = wave * 16; k0 < a.K; k0 += 64 * UN) {
    f32x4_t av[UN][MT], wv[UN][kOps][MT];
#pragma unroll
    for (int u = 0; u < UN; ++u) {
      const int k = k0 + 64 * u + 4 * fq;
#pragma unroll
      for (int j = 0; j < MT; ++j) {
        av[u][j] = load4(arow[j], k);
#pragma unroll
        for (int b = 0; b < kOps; ++b) wv[u][b][j] = load4(wrow[b][j], k);
      }
    }
#pragma unroll
    for (int u = 0; u < UN; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int b = 0; b < kOps; ++b)
#pragma unroll
          for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < MT; ++j)
              acc[b][i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[u][b][i][e], av[u][j][e], acc[b][i][j], 0, 0, 0);
  }
  // acc value v of lane l: n = 4 (l / 16) + v, m = l % 16 within its 16 x 16 block
#pragma unroll
  for (int b = 0; b < kOps; ++b)
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < MT; ++j)
        *reinterpret_cast<f32x4_t*>(&red[wave][b][16 * j + fr][16 * i + 4 * fq]) = acc[b][i][j];
  __syncthreads();
  float* out = static_cast<float*>(a.out);
  const float* bias = static_cast<const float*>(a.bias);
#pragma unroll
  for (int idx = tid; idx < kT * kT; idx += 256) {
    const int ml = idx / kT, nl = idx % kT, m = m0 + ml, n = n0 + nl;
    if (m >= a.M || n >= a.N) continue;
    float y[kOps];
#pragma unroll
    for (int b = 0; b < kOps; ++b)
      y[b] = ((red[0][b][ml][nl] + red[1][b][ml][nl]) + red[2][b][ml][nl]) + red[3][b][ml][nl];
    float* o = out + (size_t)m * a.ldo + n;
    if constexpr (EPI == kGemmStore)
      *o = y[0] + (bias != nullptr ? bias[n] : 0.f);
    else if constexpr (EPI == kGemmResidual)
      *o = *o + y[0];
    else
      *o = y[0] / (1.0f + expf(-y[0])) * y[kOps - 1];
  }
}

// ---------------------------------------------------------------------------
// Attention
// ---------------------------------------------------------------------------
// One workgroup per (token m, head h): keys 0..pos of m's row, which are the
// row's tokens m - pos .. m (a prefilled row starts at position 0).  Same
// steps as the decode attention: s = bf16(bf16(q.k) / sqrt(d)) (fp32 models
// keep the fp32 product), exact softmax, p rounded to bf16, o = T(sum p v).
template <typename T>
__global__ void __launch_bounds__(256) k_pf_attn_rows(PrefillAttn a) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  float* sc = reinterpret_cast<float*>(smem_raw);  // [capacity]
  __shared__ float red[8];
  __shared__ float part[256];
  const int m = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
  const int D = a.head_dim, nq = a.heads, g = a.heads / a.kv_heads;
  const int kvh = h / g;
  const int pos = a.pos[m];
  const int n = pos + 1;
  const T* qkv = static_cast<const T*>(a.qkv);
  const T* q = qkv + (size_t)m * a.ld + (size_t)h * D;
  const size_t koff = (size_t)nq * D + (size_t)kvh * D;
  const size_t voff = (size_t)(nq + a.kv_heads) * D + (size_t)kvh * D;
  const long long first = (long long)m - pos;
  const float scale_div = sqrtf(static_cast<float>(D));
  float lmax = -INFINITY;
  for (int j = tid; j < n; j += 256) {
    const T* k = qkv + (size_t)(first + j) * a.ld + koff;
    float s = 0.f;
    for (int c = 0; c < D; c += 8) s = dot8(Vec8<T>::load_cached(k + c), Vec8<T>::load_cached(q + c), s);
    if constexpr (sizeof(T) == 2) s = round_bf16(s);
    s = round_bf16(s / scale_div);
    sc[j] = s;
    lmax = fmaxf(lmax, s);
  }
  lmax = wave_max(lmax);
  if ((tid & 63) == 0) red[tid >> 6] = lmax;
  __syncthreads();
  const float mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  float es = 0.f;
  for (int j = tid; j < n; j += 256) es += expf(sc[j] - mx);
  es = wave_sum(es);
  __syncthreads();
  if ((tid & 63) == 0) red[4 + (tid >> 6)] = es;
  __syncthreads();
  const float inv = 1.0f / (red[4] + red[5] + red[6] + red[7]);
  for (int j = tid; j < n; j += 256) sc[j] = round_bf16(expf(sc[j] - mx) * inv);
  __syncthreads();
  // P.V: thread (c, grp) sums element c over keys grp, grp + G, ...
  const int G = 256 / D;  // D divides 256
  const int c = tid % D, grp = tid / D;
  float o = 0.f;
  for (int j = grp; j < n; j += G) o = fmaf(sc[j], Elt<T>::f(qkv[(size_t)(first + j) * a.ld + voff + c]), o);
  part[tid] = o;
  __syncthreads();
  if (tid < D) {
    float t = 0.f;
    for (int r = 0; r < G; ++r) t += part[r * D + tid];
    static_cast<T*>(a.out)[(size_t)m * nq * D + (size_t)h * D + tid] = Elt<T>::t(t);
  }
}

// Tile shapes of the MFMA attention below (keys per tile, head dim; the
// query tiles of up to 64 come from the launch's tile list).
constexpr int kAk = 64, kAd = 128;
constexpr int kAkld = kAd + 8;   // K tile row stride (elements)
constexpr int kAvld = kAd + 16;  // V tile row stride: 4 key rows of a transposing read cover 4 x 32 bytes of distinct banks

// bf16, head_dim 128: one workgroup per (tile of up to 64 queries of one row,
// head), two passes over the key tiles of 64, no score tile in LDS.
// Wave w owns queries (w / 2) * 32 ..+32 and, in every key tile, keys
// (w % 2) * 32 ..+32.  S^T = K Q^T on MFMA (keys are the A rows, queries the
// B columns), so a lane holds 16 scores of one query (its column).
//   pass 1: every score s = bf16(bf16(q.k) / sqrt(d)) (keys past the
//     query's causal limit are -inf); per lane a running max and the sum of
//     exp(s - max) rescaled as the max grows; lanes l and l ^ 32 and the two
//     key halves are then combined: the exact row max M and the sum L.
//   pass 2: the scores again, p = bf16(exp(s - M) / L) -- the reference's
//     rounding point -- and O += P V on MFMA straight from the score
//     registers: for each 16-key block the MFMA's k index runs over the keys
//     in the order the accumulator layout holds them (j 0-7 from lanes 0-31:
//     keys +0..3 and +8..11; j 8-15 from lanes 32-63: keys +4..7 and
//     +12..15), and the value operand is read in the same order from the
//     row-major V tile by transposing LDS reads.  The two key halves'
//     partial O are added at the end.
// LDS: one K tile and one V tile (36 KB), independent of the prompt length.
//
// NT > 0, for prompts of up to NT key tiles: pass 1 keeps its scores for pass
// 2, packed (they are bf16 values: 8 registers a tile and lane), in loops
// unrolled so that the registers have fixed names.  Pass 2 then reads value
// tiles alone, one barrier each, from two LDS buffers (the second lies over
// the key tile); the first is on its way during pass 1's last tile.  What
// bounds short prompts is the chain of waits, not the work.  Per layer, computed
// twice and kept: 10 tokens 14.4 -> 9.2 us, four rows of 570 tokens in all 30.3
// -> 21.0, 64 rows of 999 tokens 2,100 -> 1,497.
constexpr int kFlashLds = 2 * kAk * kAvld * 2;
static_assert(kAk * kAkld * 2 <= kAk * kAvld * 2, "the key tile fits the first value buffer");

// Workgroup order: the (KV head, query tile) pairs P = g * ntiles + t are cut
// into chunks of kFlashChunk consecutive tiles (a 1000-token prompt's tiles
// are one chunk); chunk c runs on XCD c % 8 (workgroup b runs on XCD b % 8),
// an XCD takes its chunks in order, a chunk's tiles in order, and the G
// query heads that share the KV head back to back.  The keys and values of a
// row and KV head are then read from one XCD's L2 by all of its tiles and
// heads, instead of from the memory-side cache once per head.
constexpr int kFlashChunk = 16;

constexpr int kFlashKept = 16;  // key tiles whose scores fit the registers (242 of 256)

int flash_grid(int ntiles, int heads, int kv_heads) {
  const int chunks = (ntiles * kv_heads + kFlashChunk - 1) / kFlashChunk;
  return (chunks + 7) / 8 * 8 * kFlashChunk * (heads / kv_heads);
}

// f(0), f(1), ... with the index a constant.
template <typename F, int... I>
__device__ __forceinline__ void for_each_index(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}

template <int NT>
__global__ void __launch_bounds__(256, 2) k_pf_attn_flash(PrefillAttn a, int ntiles) {
  __shared__ __align__(16) unsigned char smem[kFlashLds];
  __shared__ float stat[2][2][32][2];  // [query half][key half][query][max, sum]
  bf16_t* Ks = reinterpret_cast<bf16_t*>(smem);  // [64 keys][136]
  bf16_t* Vs = Ks + kAk * kAvld;                  // [64 keys][144]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int tix, h;
  {
    const int G = a.heads / a.kv_heads;
    const int x = blockIdx.x & 7, s = blockIdx.x >> 3;
    const int k = s / (kFlashChunk * G), rem = s - k * (kFlashChunk * G);
    const int P = (k * 8 + x) * kFlashChunk + rem / G;
    if (P >= ntiles * a.kv_heads) return;  // padding of the last chunks (uniform)
    const int g = P / ntiles;
    tix = P - g * ntiles;
    h = g * G + rem % G;
  }
  const int4 tile = a.tiles[tix];  // first query token, first token of the row, queries, first query's position
  const int m_start = tile.x, r0 = tile.y, nqt = tile.z, p0 = tile.w;
  const int nq = a.heads, kvh = h / (a.heads / a.kv_heads);
  const bf16_t* qkv = static_cast<const bf16_t*>(a.qkv);
  const size_t koff = (size_t)nq * kAd + (size_t)kvh * kAd;
  const size_t voff = (size_t)(nq + a.kv_heads) * kAd + (size_t)kvh * kAd;
  const int nkeys = p0 + nqt;
  const int nkt = (nkeys + kAk - 1) / kAk;
  const int sm = wave >> 1, sn = wave & 1, hi = lane >> 5;
  const int qloc = sm * 32 + (lane & 31);  // this lane's query within the tile
  const int qlim = p0 + qloc;              // its visible keys: j <= qlim
  constexpr float kLog2e = 1.44269504088896340736f;

  // Q fragments (B operand): query qloc (rows past the tile read the last one)
  bf16x8_t qf[kAd / 16];
  {
    const int qi = min(qloc, nqt - 1);
    const bf16_t* qrow = qkv + (size_t)(m_start + qi) * a.ld + (size_t)h * kAd + hi * 8;
#pragma unroll
    for (int ks = 0; ks < kAd / 16; ++ks) qf[ks] = lds_frag(qrow + ks * 16);
  }
  // Key tile in registers: vector v = tid + 256 i is key v / 16, elements
  // (v % 16) * 8 ..+8.  Value tile: key v % 64, elements (v / 64) * 8 ..+8.
  // Both go to LDS row-major.  Keys past the row read the last one.
  re_u32x4 kpre[4], vpre[4];
  auto load_k = [&](int kt) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int v = tid + 256 * i;
      const int tok = r0 + min(min(kt, nkt - 1) * kAk + (v >> 4), nkeys - 1);
      kpre[i] = *reinterpret_cast<const re_u32x4*>(qkv + (size_t)tok * a.ld + koff + (v & 15) * 8);
    }
  };
  auto load_v = [&](int kt, re_u32x4 (&dst)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int v = tid + 256 * i;
      const int tok = r0 + min(min(kt, nkt - 1) * kAk + (v & 63), nkeys - 1);
      dst[i] = *reinterpret_cast<const re_u32x4*>(qkv + (size_t)tok * a.ld + voff + (v >> 6) * 8);
    }
  };
  auto store_k = [&]() {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int v = tid + 256 * i;
      *reinterpret_cast<re_u32x4*>(&Ks[(v >> 4) * kAkld + (v & 15) * 8]) = kpre[i];
    }
  };
  auto store_v = [&](bf16_t* V, const re_u32x4 (&src)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int v = tid + 256 * i, key = v & 63, c = (v >> 6) * 8;
      *reinterpret_cast<re_u32x4*>(&V[key * kAvld + c]) = src[i];
    }
  };
  // This wave's K Q^T of the key tile in LDS.
  auto key_products = [&]() {
    f32x16_t acc;
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] = 0.f;
#pragma unroll
    for (int ks = 0; ks < kAd / 16; ++ks) {
      const bf16x8_t kf = lds_frag(&Ks[(sn * 32 + (lane & 31)) * kAkld + ks * 16 + hi * 8]);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[ks], acc, 0, 0, 0);
    }
    return acc;
  };
  // Scores of key tile kt for this lane's query: s[v] is key
  // kt * 64 + sn * 32 + 8 (v / 4) + 4 hi + v % 4.  MASKED: the tile reaches
  // past some query's causal limit (the tiles before nfull end at or before
  // the first query's position, so every query sees all of their keys).
  auto scores = [&](int kt, float (&sc)[16], auto masked) {
    const f32x16_t acc = key_products();
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const float x = round_bf16(div_sqrt128_bf16(round_bf16(acc[v])));
      if constexpr (decltype(masked)::value) {
        const int j = kt * kAk + sn * 32 + 8 * (v >> 2) + 4 * hi + (v & 3);
        sc[v] = j <= qlim ? x : -INFINITY;
      } else {
        sc[v] = x;
      }
    }
  };
  const int nfull = min(nkt, (p0 + 1) / kAk);

  // Pass 1: row max and sum.  A masked score adds exp2(-inf) = 0; while all
  // of a lane's scores so far are masked (m = -inf) its sum stays 0.
  float m = -INFINITY, l = 0.f;
  auto accumulate = [&](const float (&sc)[16]) {
#pragma clang fp contract(off)  // the rescaled sum is a product, then a sum
    float tmax = sc[0];
#pragma unroll
    for (int v = 1; v < 16; ++v) tmax = fmaxf(tmax, sc[v]);
    const float mn = fmaxf(m, tmax);
    const float bn = mn == -INFINITY ? 0.f : mn * kLog2e;
    float add = 0.f;
#pragma unroll
    for (int v = 0; v < 16; ++v) add += __builtin_amdgcn_exp2f(fmaf(sc[v], kLog2e, -bn));
    l = l * __builtin_amdgcn_exp2f(fmaf(m, kLog2e, -bn)) + add;
    m = mn;
  };
  auto pass1 = [&](int kt, auto masked) {
    store_k();
    load_k(kt + 1);
    lds_barrier();
    float sc[16];
    scores(kt, sc, masked);
    accumulate(sc);
    lds_barrier();
  };
  uint32_t kept[NT > 0 ? NT : 1][8];  // scores 2 i, 2 i + 1 of each key tile
  auto kept_scores = [&](const uint32_t (&k)[8], float (&sc)[16]) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      sc[2 * i] = __uint_as_float(k[i] << 16);
      sc[2 * i + 1] = __uint_as_float(k[i] & 0xffff0000u);
    }
  };
  load_k(0);
  if constexpr (NT > 0) {
    auto tile = [&](auto index) __attribute__((always_inline)) {
      constexpr int kt = decltype(index)::value;
      if (kt >= nkt) return;
      store_k();
      if (kt + 1 < nkt)
        load_k(kt + 1);
      else
        load_v(0, kpre);
      lds_barrier();
      const f32x16_t acc = key_products();
#pragma unroll
      for (int i = 0; i < 8; ++i)
        kept[kt][i] = f2_to_bf16x2_raw(div_sqrt128_bf16(round_bf16(acc[2 * i])), div_sqrt128_bf16(round_bf16(acc[2 * i + 1])));
      float sc[16];
      kept_scores(kept[kt], sc);
      if (kt >= nfull) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int j = kt * kAk + sn * 32 + 8 * (i >> 1) + 4 * hi + 2 * (i & 1);
          if (j > qlim) kept[kt][i] = (kept[kt][i] & 0xffff0000u) | 0xff80u;
          if (j + 1 > qlim) kept[kt][i] = (kept[kt][i] & 0xffffu) | 0xff800000u;
        }
        kept_scores(kept[kt], sc);
      }
      accumulate(sc);
      if (kt + 1 < nkt) lds_barrier();
    };
    for_each_index(tile, std::make_integer_sequence<int, NT>{});
    store_v(Vs, kpre);  // behind the key tile; complete at the statistics' barrier
  } else {
    int kt = 0;
    for (; kt < nfull; ++kt) pass1(kt, std::false_type{});
    for (; kt < nkt; ++kt) pass1(kt, std::true_type{});
  }
  {
    const float m2 = __shfl_xor(m, 32, 64), l2 = __shfl_xor(l, 32, 64);
    const float mm = fmaxf(m, m2);
    const float bm = mm * kLog2e;
    const float a1 = m == -INFINITY ? 0.f : l * __builtin_amdgcn_exp2f(fmaf(m, kLog2e, -bm));
    const float a2 = m2 == -INFINITY ? 0.f : l2 * __builtin_amdgcn_exp2f(fmaf(m2, kLog2e, -bm));
    m = mm;
    l = a1 + a2;
  }
  if (hi == 0) {
    stat[sm][sn][lane & 31][0] = m;
    stat[sm][sn][lane & 31][1] = l;
  }
  lds_barrier();
  float M, inv;
  {
    const float m0 = stat[sm][0][lane & 31][0], l0 = stat[sm][0][lane & 31][1];
    const float m1 = stat[sm][1][lane & 31][0], l1 = stat[sm][1][lane & 31][1];
    M = fmaxf(m0, m1);
    const float bm = M * kLog2e;
    const float a0 = m0 == -INFINITY ? 0.f : l0 * __builtin_amdgcn_exp2f(fmaf(m0, kLog2e, -bm));
    const float a1 = m1 == -INFINITY ? 0.f : l1 * __builtin_amdgcn_exp2f(fmaf(m1, kLog2e, -bm));
    const float L = a0 + a1;
    inv = L > 0.f ? 1.0f / L : 0.f;
  }
  const float base = M * kLog2e;

  // Pass 2: P V.
  f32x16_t o[4];
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int v = 0; v < 16; ++v) o[t][v] = 0.f;
  // M is finite (key 0 is visible to every query), so a masked score's
  // probability is exp2(-inf) = 0.
  auto add_values = [&](const float (&sc)[16], const bf16_t* V) {
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      float pv[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) pv[e] = __builtin_amdgcn_exp2f(fmaf(sc[8 * b + e], kLog2e, -base)) * inv;
      re_u32x4 pw;
#pragma unroll
      for (int e = 0; e < 4; ++e) pw[e] = f2_to_bf16x2(pv[2 * e], pv[2 * e + 1]);
      const bf16x8_t af = __builtin_bit_cast(bf16x8_t, pw);
      const int kb = sn * 32 + 16 * b + 4 * hi;
      // Value operand by transposing LDS reads (ds_read_b64_tr_b16): in each
      // 16-lane group, lane q + 4 r names the 8 bytes of dims 4 q .. 4 q + 3
      // of key row kb + r, and lane i receives dim i's values of the 4 keys
      // in key order -- the 4 keys lane i's MFMA column needs.
      const int gi = lane & 15, q4 = (gi & 3) * 4, rr = gi >> 2, d16 = ((lane >> 4) & 1) * 16;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const bf16_t* vr = &V[(kb + rr) * kAvld + t * 32 + d16 + q4];
        const lds_v4i16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16_ptr)vr);
        const lds_v4i16 up = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16_ptr)(vr + 8 * kAvld));
        const uint2 l2 = __builtin_bit_cast(uint2, lo), u2 = __builtin_bit_cast(uint2, up);
        const re_u32x4 bw = {l2.x, l2.y, u2.x, u2.y};
        o[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af, __builtin_bit_cast(bf16x8_t, bw), o[t], 0, 0, 0);
      }
    }
  };
  auto pass2 = [&](int kt, auto masked) {
    store_k();
    store_v(Vs, vpre);
    load_k(kt + 1);
    load_v(kt + 1, vpre);
    lds_barrier();
    float sc[16];
    scores(kt, sc, masked);
    add_values(sc, Vs);
    lds_barrier();
  };
  if constexpr (NT > 0) {
    auto tile = [&](auto index) __attribute__((always_inline)) {
      constexpr int kt = decltype(index)::value;
      if (kt >= nkt) return;
      if (kt + 1 < nkt) load_v(kt + 1, kpre);
      float sc[16];
      kept_scores(kept[kt], sc);
      add_values(sc, kt % 2 == 0 ? Vs : Ks);
      if (kt + 1 < nkt) store_v(kt % 2 == 0 ? Ks : Vs, kpre);
      lds_barrier();
    };
    for_each_index(tile, std::make_integer_sequence<int, NT>{});
  } else {
    load_k(0);
    load_v(0, vpre);
    int kt = 0;
    for (; kt < nfull; ++kt) pass2(kt, std::false_type{});
    for (; kt < nkt; ++kt) pass2(kt, std::true_type{});
  }
  // The two key halves' partial O: the sn = 1 waves hand theirs over in LDS
  // (the tiles are free now), the sn = 0 waves add (sn 0 + sn 1) and store.
  float* ox = reinterpret_cast<float*>(smem);  // [2 query halves][4][16][64]
  if (sn == 1) {
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int v = 0; v < 16; ++v) ox[((sm * 4 + t) * 16 + v) * 64 + lane] = o[t][v];
  }
  lds_barrier();
  if (sn == 0) {
    bf16_t* out = static_cast<bf16_t*>(a.out);
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int qi = sm * 32 + 8 * (v >> 2) + 4 * hi + (v & 3);
        const int col = t * 32 + (lane & 31);
        const float y = o[t][v] + ox[((sm * 4 + t) * 16 + v) * 64 + lane];
        if (qi < nqt) out[(size_t)(m_start + qi) * nq * kAd + (size_t)h * kAd + col] = f_to_bf16(y);
      }
  }
}

}  // namespace

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------
hipError_t launch_prefill_embed(const PrefillRows& a, int dtype_bytes, hipStream_t stream) {
  if (a.M <= 0) return hipSuccess;
  if (dtype_bytes == 2)
    k_pf_embed<bf16_t><<<a.M, 256, 0, stream>>>(a);
  else
    k_pf_embed<float><<<a.M, 256, 0, stream>>>(a);
  return hipGetLastError();
}

hipError_t launch_prefill_rmsnorm(void* x, const void* w, void* y, int M, int H, float eps, int dtype_bytes,
                                  const float* part, int parts, hipStream_t stream) {
  if (M <= 0) return hipSuccess;
  if (H % 8 != 0 || H > kNormRow || (parts > 0 && dtype_bytes != 2)) return hipErrorInvalidValue;
  if (parts > 0)
    k_pf_rmsnorm<bf16_t, true><<<M, 512, 0, stream>>>(x, w, y, H, eps, part, parts);
  else if (dtype_bytes == 2)
    k_pf_rmsnorm<bf16_t, false><<<M, 256, 0, stream>>>(x, w, y, H, eps, nullptr, 0);
  else
    k_pf_rmsnorm<float, false><<<M, 256, 0, stream>>>(x, w, y, H, eps, nullptr, 0);
  return hipGetLastError();
}

hipError_t launch_prefill_qkv_post(const PrefillQkv& a, int dtype_bytes, hipStream_t stream) {
  if (a.M <= 0) return hipSuccess;
  if (a.head_dim % 16 != 0 || a.ld % 8 != 0) return hipErrorInvalidValue;
  if (a.parts > 0) {
    if (dtype_bytes != 2) return hipErrorInvalidValue;
    const int vecs = (a.heads + 2 * a.kv_heads) * (a.head_dim / 16);
    k_pf_qkv_post<bf16_t, true><<<a.M, std::min(512, (vecs + 63) / 64 * 64), 0, stream>>>(a);
  } else if (dtype_bytes == 2) {
    k_pf_qkv_post<bf16_t, false><<<a.M, 256, 0, stream>>>(a);
  } else {
    k_pf_qkv_post<float, false><<<a.M, 256, 0, stream>>>(a);
  }
  return hipGetLastError();
}

template <int EPI, int MJ, int GN = kGn>
static hipError_t gemm_launch(const GemmArgs& a, int splits, hipStream_t stream) {
  constexpr int ST = gemm_stages(MJ), kLds = gemm_lds_bytes(MJ, ST, GN);
  constexpr int kTileN = EPI == kGemmSwiGlu ? GN / 2 : GN;
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(k_gemm_bf16<EPI, MJ, ST, GN>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
  if (attr != hipSuccess) return attr;
  const int nM = (a.M + gemm_tile_m(MJ) - 1) / gemm_tile_m(MJ), nN = (a.N + kTileN - 1) / kTileN;
  k_gemm_bf16<EPI, MJ, ST, GN><<<nM * nN * splits, kGthreads, kLds, stream>>>(a, nM, nN, splits);
  return hipGetLastError();
}
// Gate/up of up to 192 tokens: its tiles of 128 columns are one row of them,
// fewer than the CUs (148 of 256 at the 7B shape), and a CU takes a stage's W
// rows no faster for the idle ones.  Tiles of 96 columns where they fit the CUs
// in one round too (198): 10 tokens 54.3 -> 49.0 us, 64 tokens 61.8 -> 53.8, 65
// 66.4 -> 56.6, 128 72.4 -> 64.7, 160 99.3 -> 91.4.  256-row tiles gain nothing
// (220 tokens 100.5 and 99.7), and stay.
template <int EPI>
static hipError_t gemm_launch_mj(const GemmArgs& a, const GemmPlan& p, hipStream_t stream) {
  if constexpr (EPI == kGemmSwiGlu) {
    constexpr int kCols = kGnNarrow / 2, kCus = 256;
    if (a.M <= gemm_tile_m(p.mj) && (a.N + kCols - 1) / kCols <= kCus) {
      if (p.mj == 1) return gemm_launch<EPI, 1, kGnNarrow>(a, 1, stream);
      if (p.mj == 2) return gemm_launch<EPI, 2, kGnNarrow>(a, 1, stream);
      if (p.mj == 3) return gemm_launch<EPI, 3, kGnNarrow>(a, 1, stream);
    }
  }
  switch (p.mj) {
    case 1: return gemm_launch<EPI, 1>(a, p.splits, stream);
    case 2: return gemm_launch<EPI, 2>(a, p.splits, stream);
    case 3: return gemm_launch<EPI, 3>(a, p.splits, stream);
    default: return gemm_launch<EPI, 4>(a, p.splits, stream);
  }
}

// Three kernels by the number of tiles, so that each still gives every CU work:
// - through LDS from three tiles per CU on (SwiGLU: four), where both operands
//   can be read 16 bytes at a time, else past one per CU.  Matrix cores and LDS
//   (M x N x K): 1,000 x 2,048 x 1,024 (512 tiles) 88 and 97 us, 1,000 x 3,584 x
//   1,024 (896) 142 and 142, 16,000 x 256 x 688 (1,000) 116 and 102, 2,000 x
//   2,048 x 1,024 (1,024) 157 and 145, 4,096 x 4,096 x 1,024 596 and 479; 4-byte
//   loads, 1,000 x 1,000 x 1,023 (256) 95 and 110, 1,024 x 1,536 x 1,023 (384)
//   143 and 109, 4,096 x 4,096 x 1,023 1,413 and 503.  SwiGLU: 512 x 3,584 x
//   1,024 (896) 136 and 142, 1,000 x 2,048 x 1,024 (1,024) 148 and 146, 4,096 x
//   4,096 x 1,024 1,142 and 934 (two products, the elementwise pass not
//   counted: 960).
// - below, on the matrix cores, 32 x 32 (twice the products per byte) from two
//   workgroups per CU on, else 16 x 16 (16 x 16 against 32 x 32): 66 x 256 x 688
//   5.0 and 8.9 us, 500 x 256 x 688 6.8 and 9.2, 500 x 512 x 256 6.7 and 6.0;
//   2,044 x 256 x 688 20.0 and 15.6, 2,044 x 1,376 x 256 44.0 and 31.2.
template <int EPI>
static hipError_t gemm_f32_launch(const GemmArgs& a, hipStream_t stream) {
  constexpr unsigned kCus = 256;
  auto tiles = [&](int t) { return ((long long)a.M + t - 1) / t * (((long long)a.N + t - 1) / t); };
  const uintptr_t addr = reinterpret_cast<uintptr_t>(a.A) | reinterpret_cast<uintptr_t>(a.W) |
                         (EPI == kGemmSwiGlu ? reinterpret_cast<uintptr_t>(a.W2) : 0);
  const bool vec = (addr & 15) == 0 && a.K % 4 == 0 && a.lda % 4 == 0 && a.ldw % 4 == 0;
  constexpr unsigned kTileN = EPI == kGemmSwiGlu ? 32 : 64;
  const unsigned m_tiles = (a.M + 63u) / 64, n_tiles = (a.N + kTileN - 1) / kTileN;
  const unsigned long long lds_tiles = (unsigned long long)m_tiles * n_tiles;
  if (vec ? lds_tiles >= (EPI == kGemmSwiGlu ? 4 : 3) * kCus : lds_tiles > kCus) {
    // N tiles next to each other share A's rows in L2; a grid's second dimension holds 65,535
    const int m_on_x = m_tiles > 65535;
    k_gemm_f32_lds<EPI><<<m_on_x ? dim3(m_tiles, n_tiles) : dim3(n_tiles, m_tiles), 256, 0, stream>>>(a, m_on_x);
    return hipGetLastError();
  }
  const bool large = tiles(32) >= 2 * kCus;
  const int t = large ? 32 : 16, nN = (a.N + t - 1) / t;
  auto run = [&](auto mt, auto v) {
    k_gemm_f32<EPI, decltype(mt)::value, decltype(v)::value>
        <<<static_cast<unsigned>(tiles(t)), 256, 0, stream>>>(a, nN);
    return hipGetLastError();
  };
  using one = std::integral_constant<int, 1>;
  using two = std::integral_constant<int, 2>;
  if (large) return vec ? run(two{}, std::true_type{}) : run(two{}, std::false_type{});
  return vec ? run(one{}, std::true_type{}) : run(one{}, std::false_type{});
}

// Tile height and K ranges of a bf16 GEMM: the pair with the least estimated
// time, rounds x (K steps of a range x time per step + start and end) plus
// the partial sums' write and read.  The times are fits to one MI355X at the
// 7B projections, M = 10 .. 2,000 (steps of K = 64 with the tile's stages):
// 0.66, 0.78, 1.25 and 1.3 us a step at 64, 128, 192 and 256 rows, about 4 us
// a workgroup, partials at 2.2 TB/s through both kernels.  Ranges are taken
// only while all of them fit one round (a second round of half-filled CUs
// always lost: qkv at 120 tokens 13.3 us in 7 ranges, 20.2 in 8).  All of it is
// fitted to the whole device, so its 256 CUs are a constant here.
// Measured, 256-row tiles without ranges against the plan's choice: 10
// tokens, qkv 65 -> 9.0 us, o 65 -> 8.0, gate/up 83 -> 53, down 369 -> 26;
// 570 tokens, qkv 66 -> 30, o 66 -> 23, gate/up 171 -> 166-174, down 355 ->
// 81; from about 2,000 tokens on the 256-row tile without ranges is chosen.
GemmPlan plan_gemm(int M, int N, int K, bool swiglu, size_t part_bytes) {
  constexpr int kCus = 256;
  constexpr double kStep[4] = {0.66, 0.78, 1.25, 1.3}, kFixed = 4.0, kPartBytesPerUs = 2.2e6;
  const int steps = K / kGk, nN = (N + (swiglu ? kGn / 2 : kGn) - 1) / (swiglu ? kGn / 2 : kGn);
  GemmPlan best{4, 1};
  double best_us = 0;
  for (int mj = 4; mj >= 1; --mj) {
    const long long tiles = (long long)((M + gemm_tile_m(mj) - 1) / gemm_tile_m(mj)) * nN;
    for (int s = 1; s <= steps; ++s) {
      const size_t bytes = s > 1 ? (size_t)s * M * N * sizeof(float) : 0;
      if (s > 1 && (swiglu || tiles * s > kCus || bytes > part_bytes)) break;
      const double rounds = static_cast<double>((tiles * s + kCus - 1) / kCus);
      const double us = rounds * ((steps + s - 1) / s * kStep[mj - 1] + kFixed) + bytes / kPartBytesPerUs;
      if (best_us == 0 || us < best_us) {
        best = GemmPlan{mj, s};
        best_us = us;
      }
    }
  }
  return best;
}

hipError_t launch_gemm(const GemmArgs& a, int epi, int dtype_bytes, hipStream_t stream, GemmPlan plan) {
  if (a.M <= 0 || a.N <= 0) return hipSuccess;
  if (dtype_bytes == 2) {
    const bool swiglu = epi == kGemmSwiGlu;
    const bool aligned = ((reinterpret_cast<uintptr_t>(a.A) | reinterpret_cast<uintptr_t>(a.W) |
                           reinterpret_cast<uintptr_t>(a.out) | reinterpret_cast<uintptr_t>(swiglu ? a.W2 : a.W)) &
                          15) == 0;
    if (a.K <= 0 || a.K % kGk != 0 || a.N % 8 != 0 || a.lda % 8 != 0 || a.ldw % 8 != 0 || a.ldo % 8 != 0 ||
        !aligned || (swiglu && a.W2 == nullptr))
      return hipErrorInvalidValue;
    const GemmPlan p = plan.mj != 0 ? plan : plan_gemm(a.M, a.N, a.K, swiglu, 0);
    if (p.mj < 1 || p.mj > 4 || p.splits < 1 || p.splits > a.K / kGk || (p.splits > 1 && a.part == nullptr))
      return hipErrorInvalidValue;
    if (a.part != nullptr) return gemm_launch_mj<kGemmPart>(a, p, stream);
    if (epi == kGemmStore) return gemm_launch_mj<kGemmStore>(a, p, stream);
    if (epi == kGemmResidual) return gemm_launch_mj<kGemmResidual>(a, p, stream);
    return gemm_launch_mj<kGemmSwiGlu>(a, p, stream);
  } else {
    if (a.K <= 0 || a.part != nullptr || (epi == kGemmSwiGlu && a.W2 == nullptr)) return hipErrorInvalidValue;
    if (epi == kGemmStore) return gemm_f32_launch<kGemmStore>(a, stream);
    if (epi == kGemmResidual) return gemm_f32_launch<kGemmResidual>(a, stream);
    return gemm_f32_launch<kGemmSwiGlu>(a, stream);
  }
}

// The MFMA attention serves bf16 models with head_dim 128 (any window: its
// LDS does not depend on the prompt length).
bool prefill_attention_mfma(const Dims& d) { return d.dtype_bytes == 2 && d.head_dim == kAd; }

// Dynamic LDS of the per-(token, head) kernel: the scores of the window.
size_t prefill_attention_lds(const Dims& d, int max_keys) {
  (void)d;
  return (size_t)max_keys * sizeof(float);
}

hipError_t prepare_prefill(const Dims& d) {
  if (prefill_attention_mfma(d)) return hipSuccess;
  const int bytes = static_cast<int>(prefill_attention_lds(d, d.capacity));
  if (d.dtype_bytes == 2)
    return hipFuncSetAttribute(reinterpret_cast<const void*>(k_pf_attn_rows<bf16_t>),
                               hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  return hipFuncSetAttribute(reinterpret_cast<const void*>(k_pf_attn_rows<float>),
                             hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
}

hipError_t launch_prefill_attention(const PrefillAttn& a, const Dims& d, int ntiles, hipStream_t stream) {
  if (a.M <= 0) return hipSuccess;
  if (prefill_attention_mfma(d)) {
    if (ntiles <= 0) return hipErrorInvalidValue;
    if (d.heads % d.kv_heads != 0) return hipErrorInvalidValue;
    // The pass's longest prompt decides for all of its rows: one of more than
    // 1,024 tokens has the shorter ones compute their scores twice too, as every
    // prompt would without the kept scores (64 rows of 999 tokens, a layer:
    // 2,100 us against 1,497).
    const int grid = flash_grid(ntiles, d.heads, d.kv_heads), key_tiles = (a.max_keys + kAk - 1) / kAk;
    if (key_tiles <= 1)
      k_pf_attn_flash<1><<<grid, 256, 0, stream>>>(a, ntiles);
    else if (key_tiles <= 4)
      k_pf_attn_flash<4><<<grid, 256, 0, stream>>>(a, ntiles);
    else if (key_tiles <= kFlashKept)
      k_pf_attn_flash<kFlashKept><<<grid, 256, 0, stream>>>(a, ntiles);
    else
      k_pf_attn_flash<0><<<grid, 256, 0, stream>>>(a, ntiles);
  } else {
    if (256 % d.head_dim != 0 || d.head_dim % 8 != 0) return hipErrorInvalidValue;
    const size_t bytes = (size_t)d.capacity * sizeof(float);
    if (d.dtype_bytes == 2)
      k_pf_attn_rows<bf16_t><<<dim3(a.M, d.heads), 256, bytes, stream>>>(a);
    else
      k_pf_attn_rows<float><<<dim3(a.M, d.heads), 256, bytes, stream>>>(a);
  }
  return hipGetLastError();
}

}  // namespace re

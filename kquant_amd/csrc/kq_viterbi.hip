// SQG trellis quantizer (tail-biting Viterbi over 16-bit states) on MI355X:
// the search of kquant/csrc/qsrt_quantize_tiles_kernel.cuh with the SQG
// E4M3 labels of kquant/csrc/sqg_quantize.cu, bit for bit.
//
// A tile of 256 values is coded as 256 K-bit edges (K = 2, 3, 4); the state
// at a step is the last 16 bits of the edge stream, a node its low 16 - K
// bits, and node o is reached from nodes (o >> K) + k 2^(16-2K), k < 2^K, by
// state (k << (16-K)) | o with label lut[state].  In fp16, as the reference:
// w = fp16(x); d = fp16(label - w); the cost is fp16(d d) on a pass's first
// step (the closing pass forces its start node by +inf on every other
// predecessor), else fp16(fma(d, d, prev)) with one rounding; each node keeps
// the first predecessor with the strictly smallest cost.  A primer pass over
// positions -ctx .. ctx-1 is traced back from the argmin of its incoming cost
// buffer - which, after the buffer swaps, holds the second-to-last step's
// costs - to the node before position 0; the closing pass runs 0 .. 255 from
// that node and its traceback gives every position's state and label.  The
// argmin breaks ties as the reference's shuffle-down reductions do: smallest
// (bitrev5(e % 1024 / 32), bitrev5(e % 32), e / 1024).
//
// MI355X mapping: one workgroup per tile, persistent over the tiles.  What
// bounds the search is VALU: 2^16 edge evaluations per step and tile.
//  * Thread t owns NPT = 2^(16-K) / T consecutive nodes, so the 2^16 / T
//    labels it ever needs stay in its registers as packed fp16 (32 with 1,024
//    threads, 64 with 512): no label table in LDS and no E4M3 conversion per
//    edge, and its nodes share their predecessors (NPT / 2^K of them per k,
//    one LDS read each), whose costs both LDS buffers hold.
//  * The 2^K edge pairs of two nodes take a packed difference and fma each,
//    then a tournament of packed minima and differences whose sign bits are
//    the comparisons (costs are never negative, so their bits order as their
//    values do): the index of the winner is picked out of the sign bits at
//    the end.  (32-bit keys cost << 16 | k and min3: 1.33 ms at 448 tiles
//    against 1.25.)  Steps whose decisions are not kept (the primer's first half)
//    take the minima alone.
//  * The traceback is a chain of dependent reads of the decisions (K bits per
//    node and step in a per-workgroup global workspace): a wave reads the decisions of all nodes that the next
//    two to four steps can reach at once, so one memory latency covers them.
//  * With more tiles than CUs, 512-thread workgroups, two per CU: one tile's
//    traceback and barriers overlap the other's search.
// K = 3, ctx 128: 448 tiles 3.80 -> 1.25 ms, 164 tiles 1.95 -> 0.68 ms against
// labels looked up and converted per edge, one tile per CU and one thread's
// traceback.
//
// The same search runs against the two procedural EXL3 control codebooks of
// kquant/csrc/exl3_compat/quant/codebook.cuh (sqg_quantize.cu:261-330), whose
// label of a state is computed, not looked up (no LDS table then):
//   MCG  (1): x = state * 0xCBAC1FED mod 2^32; x = (x & 0x8fff8fff) ^ 0x3b603b60;
//             label = fp16(lo + hi), lo / hi the fp16 numbers x's two halves encode
//             (codebook.cuh:50-59, 64-79);
//   MUL1 (2): x = state * 0x83DCD12D mod 2^32; h = the fp16 1024 + (sum of x's
//             four bytes); label = fp16(h * fp16(0x1eee) + fp16(0xc931)), one
//             rounding (codebook.cuh:27-47, 80-92).
// The products of successive predecessors differ by C << (16 - K) mod 2^32,
// so each predecessor costs an add, as in qsrt_quantize_tiles_kernel.cuh:131-145.
#include "kq_internal.h"

#include <type_traits>

namespace kq {
namespace viterbi {

typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

template <int K> constexpr int edges() { return 65536 >> K; }
// decision bytes per step: K bits a node (3 take the room of 4)
template <int K> constexpr int row_bytes() { return K == 2 ? edges<K>() / 4 : edges<K>() / 2; }

// Global accesses of the table and the decisions, which a caller may hand over
// at any address (one instruction all the same).
template <typename T>
__device__ __forceinline__ T load_bytes(const uint8_t* p) {
  T v;
  __builtin_memcpy(&v, p, sizeof(T));
  return v;
}
template <typename T>
__device__ __forceinline__ void store_bytes(uint8_t* p, T v) {
  __builtin_memcpy(p, &v, sizeof(T));
}

// E4M3 (fn) byte -> fp16, exact (labels are finite).
__device__ __forceinline__ _Float16 e4m3_to_f16(uint32_t b) {
  const uint32_t s = (b >> 7) & 1, e = (b >> 3) & 15, m = b & 7;
  float v;
  if (e == 0) v = (float)m * 0.001953125f;
  else v = __builtin_bit_cast(float, ((e + 120u) << 23) | (m << 20));
  return (_Float16)(s ? -v : v);
}

// The labels of predecessor k for nodes 2p and 2p + 1, from a 16-bit
// little-endian pair of E4M3 bytes: each byte's 7 magnitude bits shifted
// left by 7 are the fp16 pattern of its value / 2^8 (E4M3 exponent bias 7
// against fp16's 15; E4M3 subnormals land on fp16 subnormals), the sign bit
// moves to bit 15, and one exact packed multiply by 2^8 finishes.
__device__ __forceinline__ h2_t pair_labels(uint32_t word16) {
  const uint32_t t = (word16 & 0xffu) | ((word16 & 0xff00u) << 8);  // bytes -> [b0, 0, b1, 0]
  const uint32_t bits = ((t & 0x007f007fu) << 7) | ((t & 0x00800080u) << 8);
  h2_t scale;
  scale[0] = (_Float16)256.0f;
  scale[1] = (_Float16)256.0f;
  return __builtin_bit_cast(h2_t, bits) * scale;
}

__device__ __forceinline__ int bitrev5(int v) { return (int)(__builtin_bitreverse32((uint32_t)v) >> 27); }

// codebook ids: 0 = an SQG E4M3 table, 1 = MCG, 2 = MUL1
template <int CB> constexpr uint32_t cb_mult() { return CB == 1 ? 0xCBAC1FEDu : 0x83DCD12Du; }

// procedural labels of states s and s + 1 from their products x0 = s C and
// x1 = x0 + C (mod 2^32)
template <int CB>
__device__ __forceinline__ h2_t procedural_pair(uint32_t x0, uint32_t x1) {
  if constexpr (CB == 1) {
    const uint32_t v0 = (x0 & 0x8fff8fffu) ^ 0x3b603b60u;
    const uint32_t v1 = (x1 & 0x8fff8fffu) ^ 0x3b603b60u;
    const uint32_t lo = (v0 & 0xffffu) | (v1 << 16);
    const uint32_t hi = (v0 >> 16) | (v1 & 0xffff0000u);
    return __builtin_bit_cast(h2_t, lo) + __builtin_bit_cast(h2_t, hi);
  } else {
    // v_sad_u8 against zero: the sum of the four bytes, plus 0x6400 (1024.0)
    const uint32_t s0 = __builtin_amdgcn_sad_u8(x0, 0u, 0x6400u);
    const uint32_t s1 = __builtin_amdgcn_sad_u8(x1, 0u, 0x6400u);
    h2_t k_inv, k_bias;
    k_inv[0] = k_inv[1] = __builtin_bit_cast(_Float16, (uint16_t)0x1eee);   // 1 / 147.7
    k_bias[0] = k_bias[1] = __builtin_bit_cast(_Float16, (uint16_t)0xc931); // -10.38
    return __builtin_elementwise_fma(__builtin_bit_cast(h2_t, (s0 & 0xffffu) | (s1 << 16)), k_inv, k_bias);
  }
}

typedef uint16_t us2_t __attribute__((ext_vector_type(2)));
typedef int16_t ss2_t __attribute__((ext_vector_type(2)));

// Minimum of N packed cost pairs and, in the top bit of each half of bit[b],
// bit b of the index of the first smallest (log2 N of them).  The bits of
// costs (never negative) order as their values do.
template <int N> struct First {
  static constexpr int BITS = N == 2 ? 1 : First<N / 2>::BITS + 1;
  uint32_t best;
  uint32_t bit[BITS];
};
template <> struct First<1> {
  static constexpr int BITS = 0;
  uint32_t best;
};

template <int N>
__device__ __forceinline__ First<N> first_smallest(const uint32_t* cost) {
  if constexpr (N == 1) {
    return First<1>{cost[0]};
  } else {
    const First<N / 2> l = first_smallest<N / 2>(cost), r = first_smallest<N / 2>(cost + N / 2);
    First<N> f;
    const us2_t a = __builtin_bit_cast(us2_t, l.best), b = __builtin_bit_cast(us2_t, r.best);
    f.best = __builtin_bit_cast(uint32_t, __builtin_elementwise_min(a, b));
    // negative where the right half's minimum is strictly smaller
    const uint32_t less = __builtin_bit_cast(uint32_t, __builtin_bit_cast(ss2_t, b) - __builtin_bit_cast(ss2_t, a));
    if constexpr (N > 2) {
#pragma unroll
      for (int i = 0; i < First<N / 2>::BITS; ++i) f.bit[i] = (less & r.bit[i]) | (~less & l.bit[i]);
    }
    f.bit[First<N>::BITS - 1] = less;
    return f;
  }
}

// The argmin order of the reference's reductions: cost first, then node e's
// place in its shuffle-down trees (14 bits, unique per node).
__device__ __forceinline__ uint32_t argmin_key(uint32_t cost_bits, int e) {
  const int t = e & 1023;
  return cost_bits << 16 | (uint32_t)((bitrev5(t >> 5) << 5 | bitrev5(t & 31)) << 4 | e >> 10);
}
__device__ __forceinline__ int argmin_node(uint32_t key) {
  const int t = (int)(key >> 4) & 1023;
  return (int)(key & 15u) << 10 | bitrev5(t >> 5) << 5 | bitrev5(t & 31);
}

template <int K, int CB, int T>
__global__ __launch_bounds__(T, 4) void sqg_viterbi_kernel(const float* __restrict__ tiles, int64_t n_tiles,
                                                           const uint8_t* __restrict__ lut, int ctx,
                                                           float* __restrict__ out_tiles,
                                                           int16_t* __restrict__ out_states,
                                                           uint8_t* __restrict__ dec_ws) {
  constexpr int E = edges<K>(), NPT = E / T, NP = NPT / 2, Q = 1 << K;
  constexpr int NIN = NPT > Q ? NPT / Q : 1;  // predecessors of a thread's nodes, per k
  constexpr int KR = 16 - K, PSTEP = 1 << (16 - 2 * K), RB = row_bytes<K>();
  constexpr uint32_t CM = cb_mult<CB>();
  static_assert(NPT >= 4 && E % T == 0, "nodes per thread");
  // A thread's decisions of one step: bit b of node 2 j + h sits in half h of
  // word NP b / 16, NP b % 16 + j places below the top; two planes of 16
  // nodes or less share a word, and four planes of 4 nodes are cut to 16 bits.
  constexpr int NW = NP * (K - 1) / 16 + 1, BYTES = RB / T;
  static_assert(BYTES == 4 * NW || (BYTES == 2 && NP * K == 8), "decision bytes per thread");
  typedef _Float16 in_t __attribute__((ext_vector_type(NIN)));
  __shared__ __attribute__((aligned(16))) _Float16 cost[2][E];
  __shared__ _Float16 w16[256];
  __shared__ uint16_t path[256];
  __shared__ uint32_t red[T / 64];
  __shared__ int sh_edge;
  const int tid = threadIdx.x;
  uint8_t* dec = dec_ws + (int64_t)blockIdx.x * 256 * RB;

  h2_t label[NP][Q];  // of nodes NPT tid + 2 j, + 1 and predecessor k
#pragma unroll
  for (int j = 0; j < NP; ++j) {
    const int o = NPT * tid + 2 * j;
#pragma unroll
    for (int k = 0; k < Q; ++k) {
      const uint32_t s = (uint32_t)(k << KR | o);
      if constexpr (CB == 0) label[j][k] = pair_labels(load_bytes<uint16_t>(lut + s));
      else label[j][k] = procedural_pair<CB>(s * CM, s * CM + CM);
    }
  }

  int cb = 0;  // cost[cb] = the buffer the next step writes; cost[cb ^ 1] its input
  // one step at position ri.  first: the pass's first step (pre_state >= 0
  // forces its predecessor); keep: write the decisions
  auto step = [&](auto first_t, auto keep_t, int ri, int pre_state) {
    constexpr bool first = decltype(first_t)::value, keep = decltype(keep_t)::value;
    cb ^= 1;  // swap: the last step's output becomes this step's input
    const _Float16* prev = cost[cb ^ 1];
    _Float16* cur = cost[cb];
    const _Float16 w = w16[ri];
    h2_t w2;
    w2[0] = w2[1] = w;
    const int in0 = NPT * tid >> K;
    in_t c[Q];
    if constexpr (!first) {
#pragma unroll
      for (int k = 0; k < Q; ++k) c[k] = *reinterpret_cast<const in_t*>(prev + in0 + k * PSTEP);
    }
    uint32_t out[NP];
    uint32_t word[NW] = {};
#pragma unroll
    for (int j = 0; j < NP; ++j) {
      const int jin = 2 * j >> K;  // which of the thread's predecessors
      auto edge = [&](int k) -> h2_t {
        const h2_t d = label[j][k] - w2;
        if constexpr (first) {
          h2_t err = d * d;
          if (pre_state >= 0 && in0 + jin + k * PSTEP != pre_state) {
            err[0] = (_Float16)__builtin_inff();
            err[1] = (_Float16)__builtin_inff();
          }
          return err;
        } else {
          h2_t c2;
          if constexpr (NIN == 1) c2[0] = c2[1] = c[k][0];
          else c2[0] = c2[1] = c[k][jin];
          return __builtin_elementwise_fma(d, d, c2);
        }
      };
      uint32_t err[Q];
#pragma unroll
      for (int k = 0; k < Q; ++k) err[k] = __builtin_bit_cast(uint32_t, edge(k));
      if constexpr (keep) {
        const First<Q> f = first_smallest<Q>(err);
        out[j] = f.best;
#pragma unroll
        for (int b = 0; b < K; ++b)
          word[NP * b / 16] |= f.bit[b] >> (NP * b % 16 + j) & 0x80008000u >> (NP * b % 16 + j);
      } else {
        us2_t best = __builtin_bit_cast(us2_t, err[0]);
#pragma unroll
        for (int k = 1; k < Q; ++k) best = __builtin_elementwise_min(best, __builtin_bit_cast(us2_t, err[k]));
        out[j] = __builtin_bit_cast(uint32_t, best);
      }
    }
    uint32_t* dst = reinterpret_cast<uint32_t*>(cur + NPT * tid);
    if constexpr (NP >= 4) {
#pragma unroll
      for (int j = 0; j < NP; j += 4)
        *reinterpret_cast<u32x4_t*>(dst + j) = u32x4_t{out[j], out[j + 1], out[j + 2], out[j + 3]};
    } else {
      *reinterpret_cast<u32x2_t*>(dst) = u32x2_t{out[0], out[1]};
    }
    if constexpr (keep) {
      uint8_t* at = dec + ri * RB + BYTES * tid;
      if constexpr (NW == 2) store_bytes(at, u32x2_t{word[0], word[1]});
      else if constexpr (BYTES == 4) store_bytes(at, word[0]);
      else store_bytes(at, (uint16_t)((word[0] >> 8 & 0xffu) | (word[0] >> 16 & 0xff00u)));
    }
    __syncthreads();
  };

  auto decision_at = [&](int ri, int e) -> int {
    const int o = e % NPT, j = o >> 1, h = o & 1;
    const uint8_t* at = dec + ri * RB + BYTES * (e / NPT);
    uint32_t half[NW];  // the halves of this parity, at bits 15 .. 0
#pragma unroll
    for (int v = 0; v < NW; ++v)
      half[v] = BYTES == 2 ? (uint32_t)at[h] << 8 : load_bytes<uint16_t>(at + 4 * v + 2 * h);
    uint32_t k = 0;
#pragma unroll
    for (int b = 0; b < K; ++b) k |= (half[NP * b / 16] >> (15 - NP * b % 16 - j) & 1u) << b;
    return (int)k;
  };

  // Walk back from `edge` through the decisions of rows - 1 .. 0 (wave 0);
  // states go to path[] when asked.  Lane l reads the decisions that steps
  // i .. i - DEPTH + 1 meet if its digits were the decisions of the first
  // DEPTH - 1 of them.
  auto trace = [&](int edge, int rows, bool keep_path) -> int {
    constexpr int DEPTH = K == 2 ? 4 : K == 3 ? 3 : 2;
    const int lane = tid & 63;
    for (int i = rows - 1; i >= 0; i -= DEPTH) {
      int b[DEPTH], e = edge;
#pragma unroll
      for (int d = 0; d < DEPTH; ++d) {
        const int ri = max(i - d, 0);
        b[d] = decision_at(ri, e);
        e = (lane >> K * d & (Q - 1)) << (16 - 2 * K) | e >> K;
      }
      int who = 0;
#pragma unroll
      for (int d = 0; d < DEPTH; ++d) {
        if (i - d < 0) break;
        const int k = __builtin_amdgcn_readlane(b[d], who);
        const int before = k << (16 - 2 * K) | edge >> K;
        if (keep_path && lane == 0) path[i - d] = (uint16_t)(before << K | edge);
        edge = before;
        who |= k << K * d;
      }
    }
    return edge;
  };

  constexpr std::true_type yes{};
  constexpr std::false_type no{};
  for (int64_t tile = blockIdx.x; tile < n_tiles; tile += gridDim.x) {
    __syncthreads();
    if (tid < 256) w16[tid] = (_Float16)tiles[tile * 256 + tid];
    __syncthreads();

    // primer: positions -ctx .. ctx - 1, decisions kept from position 0 on
    step(yes, no, 256 - ctx, -1);
    for (int i = 1; i < ctx; ++i) step(no, no, i + 256 - ctx, -1);
    for (int i = 0; i < ctx; ++i) step(no, yes, i, -1);
    // argmin of the incoming buffer (the second-to-last step's costs); edge 0 if none is finite
    {
      const uint16_t* c = reinterpret_cast<const uint16_t*>(cost[cb ^ 1]);
      uint32_t key = ~0u;
      for (int e = tid; e < E; e += T) key = min(key, argmin_key(c[e], e));
#pragma unroll
      for (int span = 32; span > 0; span >>= 1) key = min(key, (uint32_t)__shfl_xor((int)key, span));
      if ((tid & 63) == 0) red[tid >> 6] = key;
      __syncthreads();
      if (tid < 64) {
        for (int v = 0; v < T / 64; ++v) key = min(key, red[v]);
        const int edge = trace(key >= 0x7c000000u ? 0 : argmin_node(key), ctx, false);
        if (tid == 0) sh_edge = edge;
      }
    }
    __syncthreads();
    const int end_state = sh_edge;
    step(yes, yes, 0, end_state);
    for (int i = 1; i < 256; ++i) step(no, yes, i, -1);
    if (tid < 64) trace(end_state, 256, true);
    __syncthreads();
    if (tid < 256) {
      const uint32_t state = path[tid];
      out_states[tile * 256 + tid] = (int16_t)(uint16_t)state;
      if constexpr (CB == 0) out_tiles[tile * 256 + tid] = (float)e4m3_to_f16(lut[state]);
      else out_tiles[tile * 256 + tid] = (float)procedural_pair<CB>(state * CM, state * CM + CM)[0];
    }
  }
}

}  // namespace viterbi
}  // namespace kq

using namespace kq::viterbi;

extern "C" int64_t kq_sqg_quantize_workspace_size(int bits, int workgroups) {
  if (bits < 2 || bits > 4 || workgroups <= 0) return -1;
  const int64_t rb = bits == 2 ? row_bytes<2>() : bits == 3 ? row_bytes<3>() : row_bytes<4>();
  return (int64_t)workgroups * 256 * rb;
}

namespace {

// 512-thread workgroups, two per CU, once there is more than one per CU to
// run; else 1,024 threads on each tile (with one tile per CU twice the
// threads are what shortens it).
template <int K, int CB>
void launch_viterbi_k(int64_t workgroups, int cus, hipStream_t st, const float* tiles, int64_t n_tiles,
                      const uint8_t* lut, int ctx, float* out_tiles, int16_t* out_states, uint8_t* ws) {
  const unsigned grid = (unsigned)(n_tiles < workgroups ? n_tiles : workgroups);
  if ((int64_t)grid > cus)
    sqg_viterbi_kernel<K, CB, 512><<<grid, 512, 0, st>>>(tiles, n_tiles, lut, ctx, out_tiles, out_states, ws);
  else
    sqg_viterbi_kernel<K, CB, 1024><<<grid, 1024, 0, st>>>(tiles, n_tiles, lut, ctx, out_tiles, out_states, ws);
}

template <int CB>
hipError_t launch_viterbi(int bits, int64_t workgroups, hipStream_t st, const float* tiles, int64_t n_tiles,
                          const uint8_t* lut, int ctx, float* out_tiles, int16_t* out_states, uint8_t* ws) {
  int dev = 0, cus = 0;
  hipError_t e = st ? hipStreamGetDevice(st, &dev) : hipGetDevice(&dev);
  if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  if (e != hipSuccess) return e;
  auto* launch = bits == 2 ? launch_viterbi_k<2, CB> : bits == 3 ? launch_viterbi_k<3, CB> : launch_viterbi_k<4, CB>;
  launch(workgroups, cus, st, tiles, n_tiles, lut, ctx, out_tiles, out_states, ws);
  return hipGetLastError();
}

// shared checks of both entry points; 1 = nothing to do, 0 = launch, <0 = error
int check_search(const char* fn, const char* kname, const float* tiles, int64_t n_tiles, int bits,
                 int tailbite_context, float* out_tiles, int16_t* out_states, void* workspace,
                 int64_t workspace_bytes, int workgroups) {
  if (bits < 2 || bits > 4) return kq_fail(KQ_ERR_INVALID, "%s: %s supports K2--K4", fn, kname);
  if (tailbite_context < 1 || tailbite_context > 128)
    return kq_fail(KQ_ERR_INVALID, "%s: tailbite_context must be in 1..128", fn);
  if (n_tiles < 0 || workgroups <= 0) return kq_fail(KQ_ERR_INVALID, "%s: bad tile or workgroup count", fn);
  if (n_tiles == 0) return 1;
  if (!tiles || !out_tiles || !out_states || !workspace) return kq_fail(KQ_ERR_INVALID, "%s: null buffer", fn);
  if (workspace_bytes < kq_sqg_quantize_workspace_size(bits, workgroups))
    return kq_fail(KQ_ERR_INVALID, "%s: workspace too small", fn);
  return 0;
}

}  // namespace

extern "C" int kq_sqg_quantize_tiles(const float* tiles, int64_t n_tiles, const uint8_t* lut, int bits,
                                     int tailbite_context, float* out_tiles, int16_t* out_states, void* workspace,
                                     int64_t workspace_bytes, int workgroups, void* stream) {
  const char* fn = "kq_sqg_quantize_tiles";
  const int rc = check_search(fn, "SQG validation kernel", tiles, n_tiles, bits, tailbite_context, out_tiles,
                              out_states, workspace, workspace_bytes, workgroups);
  if (rc) return rc > 0 ? KQ_OK : rc;
  if (!lut) return kq_fail(KQ_ERR_INVALID, "%s: null buffer", fn);
  return kq_check_launch(launch_viterbi<0>(bits, workgroups, (hipStream_t)stream, tiles, n_tiles, lut,
                                           tailbite_context, out_tiles, out_states, (uint8_t*)workspace),
                         fn);
}

extern "C" int kq_sqg_quantize_tiles_procedural(const float* tiles, int64_t n_tiles, int bits, int codebook,
                                                int tailbite_context, float* out_tiles, int16_t* out_states,
                                                void* workspace, int64_t workspace_bytes, int workgroups,
                                                void* stream) {
  const char* fn = "kq_sqg_quantize_tiles_procedural";
  if (codebook != 1 && codebook != 2)
    return kq_fail(KQ_ERR_INVALID, "%s: procedural codebook must be 1 (MCG) or 2 (MUL1)", fn);
  const int rc = check_search(fn, "procedural control", tiles, n_tiles, bits, tailbite_context, out_tiles,
                              out_states, workspace, workspace_bytes, workgroups);
  if (rc) return rc > 0 ? KQ_OK : rc;
  auto* launch = codebook == 1 ? launch_viterbi<1> : launch_viterbi<2>;
  return kq_check_launch(launch(bits, workgroups, (hipStream_t)stream, tiles, n_tiles, nullptr, tailbite_context,
                                out_tiles, out_states, (uint8_t*)workspace),
                         fn);
}

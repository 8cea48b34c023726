// Variable-length causal attention with grouped KV heads (GQA), forward and backward, on gfx950
// fp16 MFMA with fp32 softmax statistics.
//
// Packed tokens: sequence s holds rows [cu[s], cu[s+1]); row i of a sequence attends to keys
// j <= i of the same sequence. q [N, Hq, D], k / v [N, Hkv, D] (any token / head strides, unit
// column stride), query head h reads KV head h / (Hq / Hkv); D = 128. This replaces the
// reference's per-KV-head memory-efficient attention launches (solution/unpad.py:199-294), whose
// semantics are per-row causal SDPA (solution/unpad.py:121-134).
//
// The forward is a flash-attention pass per (sequence, query tile, query heads of one KV head),
// 32 query rows of a head per wavefront, its key tiles of 64 streamed with direct-to-LDS loads and,
// where few workgroups leave the chip idle, split between two groups of wavefronts. Scores are
// computed transposed, S^T = K Q^T (v_mfma_f32_32x32x16_f16), so each lane owns one query row (its
// accumulator column): the online max / sum and the output rescale are per-lane scalars. The
// exponentiated scores are already in the B-operand layout of
// O^T = V^T P^T: the reduction over keys takes the accumulator's key order as its k-slot order,
// and V^T is read in that same order from the row-major V tile with transposing LDS reads. The
// row statistics are kept in base 2 (scores times scale * log2 e); lse is written in natural-log
// units, [Hq, N].
//
// The backward (FlashAttention-2's recurrences: P = exp(S - lse), dV = P^T dO, dP = dO V^T,
// dS = P (dP - rowsum(dO O)), dQ = scale dS K, dK = scale dS^T Q) runs as
//   attn_bwd_dot    Dd[h][t] = sum_d dO O (fp32);
//   attn_bwd_dq     per (sequence, query head, 128-row query tile): the forward's loop with
//                   dP^T = V dO^T next to S^T, and dQ^T += K^T dS^T with K^T read transposed
//                   from the K tile;
//   attn_bwd_dkdv   per (sequence, query head, 128-key tile): each lane owns a key (S and dP
//                   computed untransposed, so keys are accumulator columns), looping over
//                   64-row query tiles: dV^T += dO^T P and dK^T += Q^T dS with Q^T and dO^T read
//                   transposed from the row-major tiles; fp32 partials per query head;
//   attn_bwd_reduce the partials of a KV head's query heads summed in head order (deterministic)
//                   into dK, dV fp16.
// The dQ and dK / dV bodies run in one launch.
#include "mfma_tile.h"

#include <algorithm>

namespace talm {
namespace {

typedef uint16_t half4_t __attribute__((ext_vector_type(4)));
// 16-byte register chunks as a native vector: HIP's uint4 struct is copied with memcpy, which
// keeps a register array of them on the stack when it is stored whole into LDS.
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr int kD = 128;         // head dim
constexpr int kKeys = 64;       // keys per tile
constexpr int kKS = kD + 8;     // row stride (halfs) of a [keys][D] tile in LDS
constexpr float kLn2 = 0.693147180559945309f;

__device__ __forceinline__ float exp2_(float x) { return __builtin_amdgcn_exp2f(x); }

// The larger of lane l's and lane l ^ 32's value (v_permlane32_swap: the first result holds the
// lower half's values in both halves, the second the upper half's).
__device__ __forceinline__ float half_max(float x) {
  const uint32_t u = __builtin_bit_cast(uint32_t, x);
  const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  const uint32_t lo = r[0], hi = r[1];
  return fmaxf(__builtin_bit_cast(float, lo), __builtin_bit_cast(float, hi));
}

struct FwdArgs {
  const uint16_t* q;
  int64_t q_tok, q_head;
  const uint16_t* k;
  int64_t k_tok, k_head;
  const uint16_t* v;
  int64_t v_tok, v_head;
  const int32_t* cu;
  int group;          // query heads per KV head
  int wg_heads;       // heads per workgroup, at most H
  int head_chunks;    // workgroups per KV head (group / wg_heads)
  int list_tiles;     // > 0: the grid is list_pair's list x chunks, its sequences of at most this many tiles
  int n_seqs, chunks;
  int rank_x;         // else the grid's axes: (chunk, sequence, rank), or (rank, chunk, sequence)
  float scale_log2;   // softmax scale * log2(e)
  uint16_t* out;
  int64_t o_tok, o_head;
  float* lse;         // [Hq, n_tokens]
  int64_t n_tokens;
};

// K and V tiles of the forward in LDS: [64 keys][128 d] fp16 without padding, 16 chunks of 16
// bytes per row, chunk c of row r at position c ^ tile_swz(r). The direct-to-LDS loads write
// 1 KiB per wavefront instruction contiguously (4 rows). gfx950's LDS serves a 16-byte read in
// phases of 16 lanes over 64 four-byte banks (measured with the SQ_LDS_BANK_CONFLICT counter), so
// a 256-byte row spans every bank once and a chunk's banks depend on its position alone. The
// 4-bit key makes both reads conflict-free: the 16-byte row reads of the S = K Q^T operand
// (16 consecutive rows of one chunk per phase: the key takes 16 distinct values on them) and the
// transposing 8-byte reads (4 consecutive rows x 4 adjacent chunks per 32-lane phase: with
// r = 4a + t and c = 4b + u the position is 4 (b ^ t) + (u ^ a % 4), 16 distinct values).
constexpr int kTileBytes = kKeys * kD * 2;  // 16 KiB

__device__ __forceinline__ int tile_swz(int row) { return ((row & 3) << 2) | ((row >> 2) & 3); }
__device__ __forceinline__ int tile_chunk(int row, int chunk) { return row * 16 + (chunk ^ tile_swz(row)); }

__device__ __forceinline__ uint32_t lds_addr(const unsigned char* lds) {
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>(
      (__attribute__((address_space(3))) const unsigned char*)(lds)));
}

// LDS reads at an address plus a constant offset, as inline assembly. The compiler does not track
// them: it adds no wait for the direct-to-LDS loads in flight before them (it cannot tell that
// those write the other ring slot, and would wait for all of them), and the caller waits for the
// results itself (lgkm_wait, lgkm_wait8) before using them.
//
// ds_read_b64_tr_b16 (gfx950): within each 16-lane group, lane i receives element e (0..3) from
// row 4 e + i / 4 of the 16 x 4 matrix formed by the four halves at each lane's address, column
// i % 4 (checked on the GPU with an in-bounds probe). With lane j pointing at row K0 + j / 4,
// columns D0 + 4 (j % 4) of a row-major [keys][d] tile, lane i gets keys K0 .. K0 + 3 of column
// D0 + i: the transpose of 4 x 16 elements.
// Two of them make a 32 x 16 operand of v_mfma_f32_32x32x16_f16 transposed from a swizzled
// [rows][128] tile: A[m][k] = tile[row0 + key(k)][col0 + m], lane l holding m = l % 32 and k-slots
// 8 hh .. + 7 (hh = l / 32), whose rows follow the accumulator order of the 32-row blocks: slots
// 8 hh + e hold rows row0 + 4 hh + e (e < 4, the first read) and row0 + 8 + 4 hh + e - 4 (e >= 4, the
// second, 8 rows on). With g = l / 16 and i = l % 16 the lane points at row row0 + 4 hh + i / 4,
// columns col0 + 16 (g % 2) + 4 (i % 4) .. + 3.
__device__ __forceinline__ half4_t read_tr_untracked(uint32_t addr, int off) {
  half4_t r;
  asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(r) : "v"(addr), "n"(off));
  return r;
}
__device__ __forceinline__ half8_t read16_untracked(uint32_t addr, int off) {
  half8_t r;
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(r) : "v"(addr), "n"(off));
  return r;
}
__device__ __forceinline__ f32x4_t read_f4_untracked(uint32_t addr, int off) {
  f32x4_t r;
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(r) : "v"(addr), "n"(off));
  return r;
}
// Reads that a wait for younger ones has covered already: their registers count as written here.
__device__ __forceinline__ void lgkm_landed(f32x4_t (&r)[4]) {
  asm volatile("" : "+v"(r[0]), "+v"(r[1]), "+v"(r[2]), "+v"(r[3]));
}
// Wait until at most n LDS operations are in flight (they return in order); the registers count
// as rewritten here. n is at most 14: the counter's field has four bits, and its largest value, 15,
// means no wait.
__device__ __forceinline__ void lgkm_wait(int n, half8_t& r) {
  asm volatile("s_waitcnt lgkmcnt(%1)" : "+v"(r) : "n"(n));
}
__device__ __forceinline__ void lgkm_wait(int n, half8_t& r, half8_t& q) {
  asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(r), "+v"(q) : "n"(n));
}
__device__ __forceinline__ void lgkm_wait(int n, half4_t& r, half4_t& q) {
  asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(r), "+v"(q) : "n"(n));
}
// Wait until every LDS (and scalar-memory) operation of the wavefront has returned; the eight
// registers count as rewritten here, so no copy of them is made before the wait.
__device__ __forceinline__ void lgkm_wait8(half4_t (&r)[8]) {
  asm volatile("s_waitcnt lgkmcnt(0)"
               : "+v"(r[0]), "+v"(r[1]), "+v"(r[2]), "+v"(r[3]), "+v"(r[4]), "+v"(r[5]),
                 "+v"(r[6]), "+v"(r[7]));
}

// 16 bytes stored at byte offset `off` of the range that starts at `base`. A row past the
// sequence gets off = kOob, past the descriptor's range, and the hardware drops the store: the
// epilogues issue all their LDS reads and then all their stores, with no branch per row (a branch
// holding a read and its store made each read wait for the one before).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t store_rsrc(void* base) {
  return __builtin_amdgcn_make_buffer_rsrc(base, 0, 0x7fffffff, 0x00020000);
}
__device__ __forceinline__ void store16(__amdgpu_buffer_rsrc_t r, uint32_t off, u32x4 v) {
  __builtin_amdgcn_raw_buffer_store_b128(v, r, off, 0, 0);
}

// One [64][128] tile from global rows base[r * ld + c] (r < rows_valid, else zeros) into `dst`
// with direct-to-LDS 16-byte loads: block b (rows 4 b .. 4 b + 3) by wavefront b % W. The per-lane
// part is one register, the lane's byte offset in block `wave`: block wave + W * it lies 4 W it rows
// on (a multiple of 16 for W = 4, so its swizzle is the same), which the load takes as its scalar
// offset.
struct TileDma {
  static constexpr int W = 4, kPer = kKeys / 4 / W;
  uint32_t off, step;  // step: bytes of 4 W rows (scalar)
  int row;
  __device__ __forceinline__ void init(int64_t ld, int wave, int lane) {
    row = 4 * wave + (lane >> 4);
    off = static_cast<uint32_t>((row * ld + ((lane & 15) ^ tile_swz(row)) * 8) * 2);
    step = static_cast<uint32_t>(4 * W * ld * 2);
  }
  __device__ __forceinline__ void issue(const uint16_t* base, int rows_valid, unsigned char* dst,
                                        int wave) const {
    const __amdgpu_buffer_rsrc_t rsrc = buffer_rsrc(base);
#pragma unroll
    for (int it = 0; it < kPer; ++it)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_ptr_t)(dst + (wave + it * W) * 1024), 16,
                                               row + 4 * W * it < rows_valid ? off : kOob, it * step, 0, 0);
  }
};

// Runs body(tile, slot) for tile = 0 .. n - 1 in ring slot tile & 1, after issue(tile + 1, slot)
// put the next tile in flight into the other slot. Each tile's loads are waited for (this
// wavefront's, then the barrier for everyone's) right before its body, and the barrier also
// retires the slot the previous body read. Unrolled by two, so every slot address is a
// compile-time offset. (A third slot, two tiles in flight, measured slower.)
template <class Issue, class Body>
__device__ __forceinline__ void ring2(int n, Issue&& issue, Body&& body) {
  issue(0, 0);
  for (int t = 0; t < n; t += 2) {
    wait_vmcnt<0>();
    lds_barrier();
    if (t + 1 < n) issue(t + 1, 1);
    body(t, 0);
    if (t + 1 >= n) break;
    wait_vmcnt<0>();
    lds_barrier();
    if (t + 2 < n) issue(t + 2, 0);
    body(t + 1, 1);
  }
}

// The sum of v over the wavefront.
__device__ __forceinline__ int wave_count(int v) {
  return __builtin_amdgcn_readfirstlane(
      static_cast<int>(lanes_reduce(static_cast<uint32_t>(v), [](uint32_t x, uint32_t y) { return x + y; })));
}

// The work of up to 64 sequences, longest first: a lane holds the tiles `own` of one sequence, and the
// pairs (sequence, m), 1 <= m <= own, go by m, largest first, and within one m by sequence. Returns
// the m of pair `pair` (below the sum of own) and its sequence. C(m), the pairs with at least m, is a
// sum over the lanes, so m <= m_max is found by bisection.
constexpr int kListSeqs = 64;
__device__ __forceinline__ int list_pair(int own, int m_max, unsigned pair, int lane, int& seq) {
  int lo = 1, hi = m_max;  // the largest m with C(m) > pair
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (static_cast<unsigned>(wave_count(max(own - mid + 1, 0))) > pair) lo = mid;
    else hi = mid - 1;
  }
  const int nth = static_cast<int>(pair) - wave_count(max(own - lo, 0));
  const uint64_t has = __ballot(own >= lo);
  const bool mine = own >= lo && __popcll(has & ((uint64_t{1} << lane) - 1)) == nth;
  seq = __ffsll(static_cast<unsigned long long>(__ballot(mine))) - 1;
  return lo;
}

// Forward, one workgroup per (sequence, H query heads of one KV head, 32 * (4 / H) query rows):
// S groups of four wavefronts, each wavefront a head and 32 query rows, group g the key tiles g,
// g + S, ... of 64 keys through a two-slot ring of its own.
// Scores are computed transposed, S^T = K Q^T, so each lane owns one query row: the online
// max / sum and the output rescale are per-lane scalars, and the exponentiated scores are
// already the B operand of O^T = V^T P^T, whose A operand is read transposed from the row-major
// V tile.
// S = 1 where the grid fills the chip: two workgroups share a CU (64 KiB of LDS and at most 256
// registers each), so the two wavefronts of a SIMD belong to different workgroups and no barrier
// keeps them in step: one's softmax runs on the VALU while the other has the matrix core. What
// bounds it then: the clock, which falls from 2.4 to about 1.4 GHz with the matrix cores and the
// VALU busy together (a probe's MFMA + exponential loop), and the K / V reads from LDS.
// Against one workgroup of six or eight wavefronts per CU on 32 query rows (128 KiB of LDS, K
// operands waited for one by one): 16 rows of 128..512 tokens 36.2 -> 19.9 us, 16 of 1..1024 72.4 ->
// 39.3, [4096, 3001, 2222, 1531] 187 -> 132 us (543 -> 769 TF/s; 827 in the order of list_pair, with the
// reference maximum as below), config 2's four rows 13.7 -> 13.0.
// Not kept: the next tile's S^T issued between this one's exponentials and P V (127 against 119 us
// for 8 rows of 2048: 253 registers, the same clock), s_setprio around the MFMAs (no change).
// S = 2 where it does not: the longest workgroup's chain of key tiles sets the time (about 1.1 us
// per tile), and two groups halve it; their partial results are merged through LDS at the end.
template <int H, int S>
__global__ __launch_bounds__(256 * S, 2) void attn_fwd_kernel(FwdArgs a) {
  constexpr int R = 4 / H;           // 32-row blocks per workgroup
  constexpr int kRows = 32 * R;
  constexpr int kSlot = 2 * kTileBytes;  // one step's K and V tiles
  constexpr int kRing = 2 * kSlot;       // of one group
  constexpr int kStage = 4 * 32 * kKS * 2;  // fp16 output rows
  constexpr int kMerge = (S - 1) * 4 * (64 * 64 * 4 + 64 * 8);  // partial O, m, l per wavefront
  static_assert(S <= 2 && kMerge + kStage <= S * kRing, "merge and output staging reuse the rings");
  __shared__ __attribute__((aligned(1024))) unsigned char smem[S * kRing];

  int chunk, seq, tile;
  if (a.list_tiles) {
    const int l = threadIdx.x & 63;
    const int ll = l < a.n_seqs ? a.cu[l + 1] - a.cu[l] : 0;
    const int own = min((max(ll, 0) + kRows - 1) / kRows, a.list_tiles);
    const unsigned pair = blockIdx.x / a.chunks;
    chunk = static_cast<int>(blockIdx.x - pair * a.chunks);
    if (pair >= static_cast<unsigned>(wave_count(own))) return;
    tile = list_pair(own, a.list_tiles, pair, l, seq) - 1;
  } else {
    const int rank = static_cast<int>(a.rank_x ? blockIdx.x : blockIdx.z);
    chunk = static_cast<int>(a.rank_x ? blockIdx.y : blockIdx.x);
    seq = static_cast<int>(a.rank_x ? blockIdx.z : blockIdx.y);
    tile = (a.cu[seq + 1] - a.cu[seq] + kRows - 1) / kRows - 1 - rank;  // every sequence's longest tiles first
    if (tile < 0) return;  // the whole workgroup, before any barrier
  }
  const int kvh = chunk / a.head_chunks, hc = chunk % a.head_chunks;
  const int s0 = a.cu[seq], len = a.cu[seq + 1] - s0;
  const int q0 = tile * kRows;
  const int tid = threadIdx.x, lane = tid & 63;
  // the wavefront index in a scalar register: everything the branches, loop bounds and the
  // direct-to-LDS addresses derive from it stays wavefront-uniform
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wave = wid & 3, grp = wid >> 2;
  const int hh = lane >> 5, l32 = lane & 31;
  const int head = kvh * a.group + hc * a.wg_heads + min(wave % H, a.wg_heads - 1);
  const int w0 = q0 + 32 * (wave / H);  // the wavefront's first query row
  const int row_end = wave % H < a.wg_heads ? len : 0;  // its rows end here (a wavefront without a head: none)

  const int qrow = w0 + l32;
  const int qr = min(qrow, len - 1);
  half8_t qf[kD / 16];
  {
    const uint16_t* qp = a.q + static_cast<int64_t>(s0 + qr) * a.q_tok + head * a.q_head + 8 * hh;
#pragma unroll
    for (int s = 0; s < kD / 16; ++s) qf[s] = *reinterpret_cast<const half8_t*>(qp + 16 * s);
  }
  const int n_kt = (min(len, q0 + kRows) + kKeys - 1) / kKeys;
  const int n_steps = (n_kt + S - 1) / S;
  // tiles the wavefront's rows see: none where it has no row
  const int my_kt = w0 < row_end ? (min(len, w0 + 32) + kKeys - 1) / kKeys : 0;
  const uint16_t* kbase = a.k + static_cast<int64_t>(s0) * a.k_tok + kvh * a.k_head;
  const uint16_t* vbase = a.v + static_cast<int64_t>(s0) * a.v_tok + kvh * a.v_head;
  TileDma kd, vd;
  kd.init(a.k_tok, wave, lane);
  vd.init(a.v_tok, wave, lane);
  auto issue = [&](int step, int slot) {
    const int kt = step * S + grp;
    if (S > 1 && kt >= n_kt) return;
    unsigned char* dst = smem + grp * kRing + slot * kSlot;
    kd.issue(kbase + static_cast<int64_t>(kt * kKeys) * a.k_tok, len - kt * kKeys, dst, wave);
    vd.issue(vbase + static_cast<int64_t>(kt * kKeys) * a.v_tok, len - kt * kKeys, dst + kTileBytes,
             wave);
  };

  f32x16 o[kD / 32];
#pragma unroll
  for (int j = 0; j < kD / 32; ++j)
#pragma unroll
    for (int v = 0; v < 16; ++v) o[j][v] = 0.f;
  // m: the reference maximum of the row's scaled scores (log2 units). Past the first kEager key
  // tiles it is raised only when the row's maximum exceeds it by more than kLazy (the exponentials
  // stay <= 2^kLazy, far inside fp16, and the final O / l uses the same reference: exact up to
  // rounding). In the first tiles it follows the maximum: the weight 1 is the one that fp16 holds
  // exactly, and a short row's largest weights carry most of P's rounding error. Error of O against
  // 64 bits, lazy throughout / so / following in every tile: 16 rows of 1..1024 2.498e-4 / 2.454e-4 /
  // 2.445e-4 in 34.6 / 34.7 / 35.8 us, [4096, 3001, 2222, 1531] 2.625e-4 / 2.577e-4 / 2.547e-4 in 120.5 /
  // 122.9 / 126.8 us.
  constexpr float kLazy = 8.f;
  constexpr int kEager = 4;
  float m = -INFINITY, lsum = 0.f;
  const float c = a.scale_log2;

  // LDS addresses of the operand reads at slot 0 of the group's ring: K rows l32 of chunk 2 s + hh (s through an XOR
  // of bits 5..7), V's transposing reads of column block j (bits 6, 7), rows 4 (lane / 32) + .. and
  // 8 rows on
  const uint32_t lds0 = lds_addr(smem) + grp * kRing;
  uint32_t kaddr[kD / 16], vlo[kD / 32], vhi[kD / 32];
#pragma unroll
  for (int s = 0; s < kD / 16; ++s) kaddr[s] = lds0 + tile_chunk(l32, 2 * s + hh) * 16;
  {
    const int g = lane >> 4, i = lane & 15;
#pragma unroll
    for (int j = 0; j < kD / 32; ++j) {
      const int col = 32 * j + 16 * (g & 1) + 4 * (i & 3), row = 4 * (g >> 1) + (i >> 2);
      vlo[j] = lds0 + tile_chunk(row, col >> 3) * 16 + (col & 7) * 2;
      vhi[j] = lds0 + tile_chunk(row + 8, col >> 3) * 16 + (col & 7) * 2;
    }
  }
  auto body = [&](int step, auto slot_) __attribute__((always_inline)) {
    constexpr int kOff = decltype(slot_)::value * kSlot;
    const int kt = step * S + grp;
    if (kt >= my_kt) return;  // every key of the tile is after every row of the wavefront
    const int k0 = kt * kKeys;
    // S^T: the second 32 keys' operand reads are issued one by one behind the first block's MFMAs
    f32x16 st[2];
    half8_t kf[kD / 16];
#pragma unroll
    for (int s = 0; s < kD / 16; ++s) kf[s] = read16_untracked(kaddr[s], kOff);
#pragma unroll
    for (int b = 0; b < 2; ++b) {
#pragma unroll
      for (int v = 0; v < 16; ++v) st[b][v] = 0.f;
#pragma unroll
      for (int s = 0; s < kD / 16; ++s) {
        lgkm_wait(b == 0 ? 7 : 7 - s, kf[s]);
        st[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[s], qf[s], st[b], 0, 0, 0);
        if (b == 0) {
          __builtin_amdgcn_sched_barrier(0);
          kf[s] = read16_untracked(kaddr[s], kOff + 8192);
        }
      }
    }
    if (k0 + kKeys - 1 > w0 || k0 + kKeys > len) {  // uniform: the diagonal and the last tile
      const int lim = qr - k0 - 4 * hh;
      asm volatile("");
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int v = 0; v < 16; ++v)
          st[b][v] = 32 * b + 8 * (v >> 2) + (v & 3) > lim ? -INFINITY : st[b][v];
    }
    float mt = -INFINITY;
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int v = 0; v < 16; ++v) mt = fmaxf(mt, st[b][v]);
    mt = c * half_max(mt);
    const bool grow = mt > m + (kt < kEager ? 0.f : kLazy);
    if (__ballot(grow)) {  // some row's maximum moved: rescale those rows
      asm volatile("");
      const float m_new = grow ? mt : m;
      const float alpha = exp2_(m - m_new);  // 0 on the first tile (m = -inf), 1 if unchanged
      m = m_new;
      lsum *= alpha;
#pragma unroll
      for (int j = 0; j < kD / 32; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) o[j][v] *= alpha;
    }
    half4_t vt[2][8];
    auto read_v = [&](int g16, int buf) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < kD / 32; ++j) {
        vt[buf][2 * j] = read_tr_untracked(vlo[j], kOff + kTileBytes + g16 * 4096);
        vt[buf][2 * j + 1] = read_tr_untracked(vhi[j], kOff + kTileBytes + g16 * 4096);
      }
    };
    read_v(0, 0);
    float ps = 0.f;
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const float pv = exp2_(__builtin_fmaf(st[b][v], c, -m));
        st[b][v] = pv;
        ps += pv;
      }
    lsum += ps;
#pragma unroll
    for (int g16 = 0; g16 < 4; ++g16) {
      const int b = g16 >> 1, h = g16 & 1, buf = g16 & 1;
      lgkm_wait8(vt[buf]);  // group g16's reads have returned
      if (g16 < 3) read_v(g16 + 1, buf ^ 1);  // the next group's fly during these MFMAs
      half8_t pb;
#pragma unroll
      for (int e = 0; e < 8; ++e) pb[e] = static_cast<_Float16>(st[b][8 * h + e]);
#pragma unroll
      for (int j = 0; j < kD / 32; ++j)
        o[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
            __builtin_bit_cast(half8_t, __builtin_shufflevector(vt[buf][2 * j], vt[buf][2 * j + 1],
                                                                0, 1, 2, 3, 4, 5, 6, 7)),
            pb, o[j], 0, 0, 0);
    }
  };
  ring2(n_steps, issue, [&](int step, int slot) __attribute__((always_inline)) {
    if (slot) body(step, std::integral_constant<int, 1>{});
    else body(step, std::integral_constant<int, 0>{});
  });
  lsum += __shfl_xor(lsum, 32, kWave);  // the row's sum over both halves of the lanes
  __syncthreads();  // every wavefront is done with the tiles
  if constexpr (S > 1) {  // group 1 leaves its (m, l, O) in LDS, group 0 merges
    float* po = reinterpret_cast<float*>(smem) + wave * 64 * 64;
    float* pml = reinterpret_cast<float*>(smem) + 4 * 64 * 64 + wave * 64 * 2;
    if (grp > 0) {
#pragma unroll
      for (int j = 0; j < kD / 32; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) po[(16 * j + v) * 64 + lane] = o[j][v];
      pml[2 * lane] = m;
      pml[2 * lane + 1] = lsum;
    }
    __syncthreads();
    if (grp > 0) return;  // no barrier follows
    const float m2 = pml[2 * lane], l2 = pml[2 * lane + 1];
    const float m_new = fmaxf(m, m2);  // m is finite: group 0 has key tile 0
    const float a1 = exp2_(m - m_new);
    const float a2 = exp2_(m2 - m_new);  // 0 when group 1 had no tile (m2 = -inf)
    m = m_new;
    lsum = lsum * a1 + l2 * a2;
#pragma unroll
    for (int j = 0; j < kD / 32; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) o[j][v] = o[j][v] * a1 + po[(16 * j + v) * 64 + lane] * a2;
  }

  // O = O^T / l through LDS: each wavefront stages its 32 rows x D, then 16-byte row stores
  const float inv = 1.f / lsum;
  uint16_t* os = reinterpret_cast<uint16_t*>(smem + kMerge) + wave * 32 * kKS;
#pragma unroll
  for (int j = 0; j < kD / 32; ++j)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int d0 = 32 * j + 8 * g + 4 * hh;
      uint2 w;
      w.x = pack2(o[j][4 * g] * inv, o[j][4 * g + 1] * inv);
      w.y = pack2(o[j][4 * g + 2] * inv, o[j][4 * g + 3] * inv);
      *reinterpret_cast<uint2*>(&os[l32 * kKS + d0]) = w;
    }
  if (hh == 0 && qrow < row_end)
    a.lse[static_cast<int64_t>(head) * a.n_tokens + s0 + qrow] = (m + __log2f(lsum)) * kLn2;
  // the wavefront reads back its own staging rows: its LDS writes complete first
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  constexpr int kOut = (32 * kD / 8) / 64;
  u32x4 ov[kOut];
#pragma unroll
  for (int it = 0; it < kOut; ++it) {
    const int cc16 = it * 64 + lane, r = cc16 / (kD / 8), cc = cc16 % (kD / 8);
    ov[it] = *reinterpret_cast<const u32x4*>(&os[r * kKS + 8 * cc]);
  }
  const __amdgpu_buffer_rsrc_t ors =
      store_rsrc(a.out + static_cast<int64_t>(s0 + w0) * a.o_tok + head * a.o_head);
#pragma unroll
  for (int it = 0; it < kOut; ++it) {
    const int cc16 = it * 64 + lane, r = cc16 / (kD / 8), cc = cc16 % (kD / 8);
    store16(ors, w0 + r < row_end ? static_cast<uint32_t>((r * a.o_tok + 8 * cc) * 2) : kOob, ov[it]);
  }
}

// ------------------------------------------------------------------------------------------
// Backward
// ------------------------------------------------------------------------------------------
struct BwdArgs {
  const uint16_t* q;
  int64_t q_tok, q_head;
  const uint16_t* k;
  int64_t k_tok, k_head;
  const uint16_t* v;
  int64_t v_tok, v_head;
  const uint16_t* o;
  int64_t o_tok, o_head;
  const uint16_t* dout;
  int64_t do_tok, do_head;
  const float* lse;    // [Hq, n_tokens], natural log
  const int32_t* cu;
  int group, n_q_heads, n_kv_heads;
  int n_tiles;         // tiles per sequence (of the longest)
  float scale, scale_log2;
  int64_t n_tokens;
  float* dd;           // [Hq, n_tokens]: rowsum(dO * O)
  float* lse2;         // [Hq, n_tokens]: lse in base-2 units (lse * log2 e)
  unsigned* counter;   // the next work item of attn_bwd_queue_kernel (null: one workgroup per item)
  unsigned queue_wgs;  // its workgroups, each starting with the item of its own index
  int n_seqs;
  float* dk_part;      // [Hq, n_tokens, D] fp32
  float* dv_part;      // [Hq, n_tokens, D] fp32
  uint16_t* dq;
  int64_t dq_tok, dq_head;
  uint16_t* dk;
  int64_t dk_tok, dk_head;
  uint16_t* dv;
  int64_t dv_tok, dv_head;
  // the rotary embedding's backward folded into the outputs (null: none): cos / sin fp32
  // [n_tokens][cs_tok], and every 128-wide head of dq and dk is rotated back on its (d, d + 64)
  // pairs: dx1 = dy1 c1 + dy2 s2, dx2 = dy2 c2 - dy1 s1 (solution/rope.py:145-157)
  const float* cos;
  const float* sin;
  int64_t cs_tok;
};

// The rotary embedding's backward on one (d, d + 64) pair of four columns each: x = dy at
// columns d .. d + 3, y at d + 64 .. d + 67, of the token whose cos / sin rows are cr / sr.
__device__ __forceinline__ void rope_back4(float (&x)[4], float (&y)[4], const float* cr,
                                          const float* sr, int d) {
  const float4 c1 = *reinterpret_cast<const float4*>(cr + d);
  const float4 c2 = *reinterpret_cast<const float4*>(cr + d + kD / 2);
  const float4 s1 = *reinterpret_cast<const float4*>(sr + d);
  const float4 s2 = *reinterpret_cast<const float4*>(sr + d + kD / 2);
  const float cc1[4] = {c1.x, c1.y, c1.z, c1.w}, cc2[4] = {c2.x, c2.y, c2.z, c2.w};
  const float ss1[4] = {s1.x, s1.y, s1.z, s1.w}, ss2[4] = {s2.x, s2.y, s2.z, s2.w};
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float a = x[e], b = y[e];
    x[e] = a * cc1[e] + b * ss2[e];
    y[e] = b * cc2[e] - a * ss1[e];
  }
}

// Dd[h][t] = sum_d dO[t][h][d] * O[t][h][d] and lse2[h][t] = lse[h][t] log2 e (the exponent offset
// both backward bodies subtract): 16 lanes per (token, head), 8 columns each.
__global__ __launch_bounds__(256) void attn_bwd_dot_kernel(BwdArgs a) {
  const int64_t row = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) >> 4;  // t * Hq + h
  const int sub = threadIdx.x & 15;
  if (a.counter && blockIdx.x == 0 && threadIdx.x == 0) *a.counter = a.queue_wgs;
  const int64_t rows = a.n_tokens * a.n_q_heads;
  const int64_t r = row < rows ? row : rows - 1;
  const int64_t t = r / a.n_q_heads;
  const int h = static_cast<int>(r % a.n_q_heads);
  const u32x4 x = *reinterpret_cast<const u32x4*>(a.o + t * a.o_tok + h * a.o_head + 8 * sub);
  const u32x4 y = *reinterpret_cast<const u32x4*>(a.dout + t * a.do_tok + h * a.do_head + 8 * sub);
  float acc = lo_f(x.x) * lo_f(y.x) + hi_f(x.x) * hi_f(y.x) + lo_f(x.y) * lo_f(y.y) +
              hi_f(x.y) * hi_f(y.y) + lo_f(x.z) * lo_f(y.z) + hi_f(x.z) * hi_f(y.z) +
              lo_f(x.w) * lo_f(y.w) + hi_f(x.w) * hi_f(y.w);
#pragma unroll
  for (int off = 8; off >= 1; off >>= 1) acc += __shfl_xor(acc, off, 16);
  if (sub == 0 && row < rows) {
    const int64_t i = static_cast<int64_t>(h) * a.n_tokens + t;
    a.dd[i] = acc;
    a.lse2[i] = a.lse[i] * 1.44269504088896341f;
  }
}

// The dQ and dK / dV bodies below stream their tiles with the forward's direct-to-LDS loads into
// the swizzled [64][128] layout (tile_chunk): 16-byte row reads give the operands taken row by
// row, and the transposing reads give K^T, Q^T and dO^T straight from the same tiles, so no
// transposed copy is written.
//
// Both walk their tiles in blocks of 32 rows, software-pipelined by hand: the products that need a
// block's P and dS run one block behind its scores, so the exponentials of one block issue between
// the MFMAs of another, and every operand is read from LDS into the register its last use has just
// left, waited for with a counted lgkmcnt. The products of a tile's last block therefore still read
// it while the next tile's scores run: a three-slot ring, one tile ahead.
// What bounds them: one wavefront per SIMD (364 registers in attn_bwd_kernel; 442 and 30 spilled
// scalars in attn_bwd_queue_kernel). An unmasked 64-row step of dK / dV is about 600 instructions and
// takes 4440 cycles against 2048 of MFMAs, a 64-key step of dQ about 460 in 2940 against 1536 (clock
// stamps); taking the MFMAs out saves only 5%. In dK / dV a block's exponentials all stand beside
// the MFMAs of the products, none beside those of the scores. Against scores,
// exponentials and products one after the other with the operands read in batches (465
// registers): backward of lengths [4096, 3001, 2222, 1531] 610 -> 538 us, of 16 rows of 128..512
// 100.6 -> 94.6, of config 2's four rows 37.6 -> 35.0.
constexpr int kBwdSlot = 2 * kTileBytes + 2048;  // two tiles (+ per-wavefront lse / Dd rows: dK / dV)
constexpr int kBwdLds = 3 * kBwdSlot;

// LDS addresses of a lane's operand reads: the 16-byte reads of row l32, chunks 2 s + hh, in the slot
// the row side is at, and the transposing reads of column block j (rows 4 hh + .. and 8 rows on) in
// the slot the transposed side is at, which follows behind. A block's rows (8 KiB), a 16-row group
// (4 KiB) and the second tile are constant offsets.
struct BwdReads {
  uint32_t row[kD / 16], tlo[kD / 32], thi[kD / 32];
  __device__ __forceinline__ void init(uint32_t lds, int lane) {
    const int hh = lane >> 5, l32 = lane & 31, g = lane >> 4, i = lane & 15;
#pragma unroll
    for (int s = 0; s < kD / 16; ++s) row[s] = lds + tile_chunk(l32, 2 * s + hh) * 16;
#pragma unroll
    for (int j = 0; j < kD / 32; ++j) {
      const int col = 32 * j + 16 * (g & 1) + 4 * (i & 3), r = 4 * (g >> 1) + (i >> 2);
      tlo[j] = lds + tile_chunk(r, col >> 3) * 16 + (col & 7) * 2;
      thi[j] = lds + tile_chunk(r + 8, col >> 3) * 16 + (col & 7) * 2;
    }
  }
  __device__ __forceinline__ void next_row(uint32_t step) {
#pragma unroll
    for (int s = 0; s < kD / 16; ++s) row[s] += step;
  }
  __device__ __forceinline__ void next_t(uint32_t step) {
#pragma unroll
    for (int j = 0; j < kD / 32; ++j) {
      tlo[j] += step;
      thi[j] += step;
    }
  }
};
__device__ __forceinline__ half8_t pair8(half4_t lo, half4_t hi) {
  return __builtin_bit_cast(half8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}
// From one ring slot to the next, in bytes.
__device__ __forceinline__ uint32_t slot_step(int slot) {
  return slot == 2 ? static_cast<uint32_t>(-2 * kBwdSlot) : static_cast<uint32_t>(kBwdSlot);
}

// dQ: the forward's structure, one query row per lane (S^T = K Q^T, dP^T = V dO^T, then
// dQ^T += K^T dS^T with K^T read transposed from the K tile); `tile` is the 32W-row query tile.
template <int W, class Done>
__device__ __forceinline__ void attn_bwd_dq(const BwdArgs& a, int seq, int head, int tile,
                                            unsigned char* smem, Done&& done) {
  constexpr int kRows = 32 * W;
  const int s0 = a.cu[seq], len = a.cu[seq + 1] - s0;
  const int q0 = tile * kRows;
  if (q0 >= len) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hh = lane >> 5, l32 = lane & 31;
  const int kvh = head / a.group;
  const int qrow = q0 + 32 * wave + l32;
  const int qr = min(qrow, len - 1);
  half8_t qf[kD / 16], df[kD / 16];
  {
    const uint16_t* qp = a.q + static_cast<int64_t>(s0 + qr) * a.q_tok + head * a.q_head + 8 * hh;
    const uint16_t* dp = a.dout + static_cast<int64_t>(s0 + qr) * a.do_tok + head * a.do_head + 8 * hh;
#pragma unroll
    for (int s = 0; s < kD / 16; ++s) {
      qf[s] = *reinterpret_cast<const half8_t*>(qp + 16 * s);
      df[s] = *reinterpret_cast<const half8_t*>(dp + 16 * s);
    }
  }
  const float lse2 = a.lse2[static_cast<int64_t>(head) * a.n_tokens + s0 + qr];
  const float ddr = a.dd[static_cast<int64_t>(head) * a.n_tokens + s0 + qr];
  const int wq0 = q0 + 32 * wave;  // the wavefront's first query row

  const int n_kt = (min(len, q0 + kRows) + kKeys - 1) / kKeys;
  const int my_kt = (min(len, wq0 + 32) + kKeys - 1) / kKeys;  // tiles the wavefront's rows see
  const int lim = min(qrow, len - 1) - 4 * hh;  // a lane's last key, minus its half's offset
  const uint16_t* kbase = a.k + static_cast<int64_t>(s0) * a.k_tok + kvh * a.k_head;
  const uint16_t* vbase = a.v + static_cast<int64_t>(s0) * a.v_tok + kvh * a.v_head;
  TileDma kd, vd;
  kd.init(a.k_tok, wave, lane);
  vd.init(a.v_tok, wave, lane);
  auto issue = [&](int kt, int slot) __attribute__((always_inline)) {
    unsigned char* dst = smem + slot * kBwdSlot;
    const int r0 = kt * kKeys;
    kd.issue(kbase + static_cast<int64_t>(r0) * a.k_tok, len - r0, dst, wave);
    vd.issue(vbase + static_cast<int64_t>(r0) * a.v_tok, len - r0, dst + kTileBytes, wave);
  };

  BwdReads rd;
  rd.init(lds_addr(smem), lane);
  f32x16 acc[kD / 32], st[2], dpt[2];  // block b's scores and dP in st[b], dpt[b]
#pragma unroll
  for (int j = 0; j < kD / 32; ++j)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[j][v] = 0.f;
  half8_t sb[2];     // dS^T of the block in hand, packed: 16 keys each
  half4_t kt_[16];   // its K^T operands: [16-key group][column block][8-key halves]
  // dS^T = P^T (dP^T - Dd), P^T = exp2(S^T scale log2e - lse2): value v of block b
  auto value = [&](int b, int v) __attribute__((always_inline)) {
    const float p = exp2_(__builtin_fmaf(st[b][v], a.scale_log2, -lse2));
    sb[v >> 3][v & 7] = static_cast<_Float16>(p * (dpt[b][v] - ddr));
  };
  // ... 0 where masked, for the block whose first key is kb: only on a block that reaches past the
  // wavefront's first row or past the sequence (a uniform branch that holds no MFMA: with two
  // copies of the products the accumulators were moved between them)
  auto mask = [&](int kb) __attribute__((always_inline)) {
    if (kb + 31 > wq0 || kb + 32 > len) {
      int last = lim - kb;
      asm volatile("" : "+v"(last));  // a real branch: selects on it cannot be hoisted out
#pragma unroll
      for (int v = 0; v < 16; ++v)
        sb[v >> 3][v & 7] = 8 * (v >> 2) + (v & 3) <= last ? sb[v >> 3][v & 7] : static_cast<_Float16>(0.f);
    }
  };
  auto read_kt = [&](auto blk, int i) __attribute__((always_inline)) {  // pair i: group i / 4, block i % 4
    constexpr int kB = decltype(blk)::value;
    kt_[2 * i] = read_tr_untracked(rd.tlo[i & 3], kB * 8192 + (i >> 2) * 4096);
    kt_[2 * i + 1] = read_tr_untracked(rd.thi[i & 3], kB * 8192 + (i >> 2) * 4096);
  };
  // block kB of the tile at the row addresses: S^T and dP^T; beside the MFMAs (kPrev) the values of
  // the block before it, in the second half its K^T operand reads
  auto scores = [&](auto blk, auto prev) __attribute__((always_inline)) {
    constexpr int kB = decltype(blk)::value;
    constexpr bool kPrev = decltype(prev)::value;
    half8_t f[8];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      f[2 * s] = read16_untracked(rd.row[s], kB * 8192);
      f[2 * s + 1] = read16_untracked(rd.row[s], kTileBytes + kB * 8192);
    }
#pragma unroll
    for (int v = 0; v < 16; ++v) st[kB][v] = dpt[kB][v] = 0.f;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const int x = 2 * (s & 3);
      // outstanding behind the operand: the other row reads (8 while s < 4) and, from s = 5 on, 4
      // K^T reads per step
      lgkm_wait(s < 4 ? 7 : (7 - 2 * (s - 4)) + (kPrev ? 4 * (s - 4) : 0), f[x]);
      st[kB] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f[x], qf[s], st[kB], 0, 0, 0);
      if constexpr (kPrev) value(kB ^ 1, 2 * s);
      __builtin_amdgcn_sched_barrier(0);
      lgkm_wait(s < 4 ? 6 : (6 - 2 * (s - 4)) + (kPrev ? 4 * (s - 4) : 0), f[x + 1]);
      dpt[kB] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f[x + 1], df[s], dpt[kB], 0, 0, 0);
      if constexpr (kPrev) value(kB ^ 1, 2 * s + 1);
      __builtin_amdgcn_sched_barrier(0);
      if (s < 4) {
        f[x] = read16_untracked(rd.row[s + 4], kB * 8192);
        f[x + 1] = read16_untracked(rd.row[s + 4], kTileBytes + kB * 8192);
      } else if constexpr (kPrev) {
        read_kt(std::integral_constant<int, kB ^ 1>{}, 2 * (s - 4));
        read_kt(std::integral_constant<int, kB ^ 1>{}, 2 * (s - 4) + 1);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // dQ^T[d][q] += K^T[d][key] dS^T[key][q] of the block in hand, in the accumulator's key order
  auto gather = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      lgkm_wait(14 - 2 * i, kt_[2 * i], kt_[2 * i + 1]);
      acc[i & 3] = __builtin_amdgcn_mfma_f32_32x32x16_f16(pair8(kt_[2 * i], kt_[2 * i + 1]),
                                                          sb[i >> 2], acc[i & 3], 0, 0, 0);
    }
  };
  using B0 = std::integral_constant<int, 0>;
  using B1 = std::integral_constant<int, 1>;
  int slot = 0;  // of the tile in hand
  issue(0, 0);
  auto arrive = [&](int t) __attribute__((always_inline)) {
    wait_vmcnt<0>();
    lds_barrier();  // tile t has landed; everyone is done with tile t - 2, whose slot takes t + 1
    if (t + 1 < n_kt) issue(t + 1, slot == 2 ? 0 : slot + 1);
  };
  auto leave = [&]() __attribute__((always_inline)) {
    rd.next_row(slot_step(slot));
    slot = slot == 2 ? 0 : slot + 1;
  };
  arrive(0);
  scores(B0{}, std::false_type{});
  scores(B1{}, std::true_type{});
  mask(0);
  gather();
  leave();
  for (int t = 1; t < my_kt; ++t) {
    arrive(t);
    scores(B0{}, std::true_type{});  // block 1 of tile t - 1: never masked, a later tile is live
    gather();
    rd.next_t(slot_step(slot == 0 ? 2 : slot - 1));
    scores(B1{}, std::true_type{});
    mask(t * kKeys);
    gather();
    leave();
  }
  // the last block: nothing to run beside it (no read is in flight here; the wait says so to a
  // reader of the code in layout order too)
  asm volatile("s_waitcnt lgkmcnt(0)" : "+a"(st[1]), "+a"(dpt[1]));
#pragma unroll
  for (int i = 0; i < 8; ++i) read_kt(B1{}, i);
#pragma unroll
  for (int v = 0; v < 16; ++v) value(1, v);
  mask((my_kt - 1) * kKeys + 32);
  gather();
  for (int t = my_kt; t < n_kt; ++t) {  // tiles that only later rows of the workgroup see
    arrive(t);
    slot = slot == 2 ? 0 : slot + 1;
  }

  done();
  __syncthreads();  // every wavefront is done with the ring: it becomes the output staging
  uint16_t* os = reinterpret_cast<uint16_t*>(smem) + wave * 32 * kKS;
  // dQ = scale * the accumulated sum; rows d = 32 j + 8 g + 4 hh + e of block j pair with the
  // same (g, e) of block j + 2 (d + 64): with cos / sin the rotary backward is applied in fp32
  // here, before the one rounding to fp16 (row qr: rows past the sequence are not stored)
  float dqv[kD / 32][16];
#pragma unroll
  for (int j = 0; j < kD / 32; ++j)
#pragma unroll
    for (int v = 0; v < 16; ++v) dqv[j][v] = acc[j][v] * a.scale;
  if (a.cos) {
    const float* cr = a.cos + static_cast<int64_t>(s0 + qr) * a.cs_tok;
    const float* sr = a.sin + static_cast<int64_t>(s0 + qr) * a.cs_tok;
#pragma unroll
    for (int j = 0; j < kD / 64; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        float x[4], y[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          x[e] = dqv[j][4 * g + e];
          y[e] = dqv[j + 2][4 * g + e];
        }
        rope_back4(x, y, cr, sr, 32 * j + 8 * g + 4 * hh);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          dqv[j][4 * g + e] = x[e];
          dqv[j + 2][4 * g + e] = y[e];
        }
      }
  }
#pragma unroll
  for (int j = 0; j < kD / 32; ++j)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int d0 = 32 * j + 8 * g + 4 * hh;
      uint2 w;
      w.x = pack2(dqv[j][4 * g], dqv[j][4 * g + 1]);
      w.y = pack2(dqv[j][4 * g + 2], dqv[j][4 * g + 3]);
      *reinterpret_cast<uint2*>(&os[l32 * kKS + d0]) = w;
    }
  // the wavefront reads back its own staging rows: its LDS writes complete first
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  constexpr int kOut = (32 * kD / 8) / 64;  // 16-byte chunks per lane
  u32x4 ov[kOut];
#pragma unroll
  for (int it = 0; it < kOut; ++it) {
    const int c = it * 64 + lane, r = c / (kD / 8), cc = c % (kD / 8);
    ov[it] = *reinterpret_cast<const u32x4*>(&os[r * kKS + 8 * cc]);
  }
  const __amdgpu_buffer_rsrc_t ors =
      store_rsrc(a.dq + static_cast<int64_t>(s0 + wq0) * a.dq_tok + head * a.dq_head);
#pragma unroll
  for (int it = 0; it < kOut; ++it) {
    const int c = it * 64 + lane, r = c / (kD / 8), cc = c % (kD / 8);
    store16(ors, wq0 + r < len ? static_cast<uint32_t>((r * a.dq_tok + 8 * cc) * 2) : kOob, ov[it]);
  }
}

// dK / dV partials of one query head; `tile` is the 32W-key tile, each lane owns one key (S and
// dP untransposed: keys are accumulator columns), looping over 64-row query tiles: dV^T += dO^T P
// and dK^T += Q^T dS with Q^T and dO^T read transposed from the row-major tiles. Each slot holds
// the Q tile, the dO tile, then each wavefront's copy of the tile's 64 lse and 64 Dd values.
template <int W, class Done>
__device__ __forceinline__ void attn_bwd_dkdv(const BwdArgs& a, int seq, int head, int tile,
                                              unsigned char* smem, Done&& done) {
  constexpr int kCols = 32 * W;  // keys per workgroup
  constexpr int kRowsT = kKeys;  // query rows per tile
  const int s0 = a.cu[seq], len = a.cu[seq + 1] - s0;
  const int k0 = tile * kCols;
  if (k0 >= len) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hh = lane >> 5, l32 = lane & 31;
  const int kvh = head / a.group;
  const int key = k0 + 32 * wave + l32;
  const int kr_ = min(key, len - 1);
  const int wk0 = k0 + 32 * wave;  // the wavefront's first key
  const int q_end = key < len ? len : 0;  // a lane's query rows end here (a key past the sequence: none)
  half8_t kf[kD / 16], vf[kD / 16];
  {
    const uint16_t* kp = a.k + static_cast<int64_t>(s0 + kr_) * a.k_tok + kvh * a.k_head + 8 * hh;
    const uint16_t* vp = a.v + static_cast<int64_t>(s0 + kr_) * a.v_tok + kvh * a.v_head + 8 * hh;
#pragma unroll
    for (int s = 0; s < kD / 16; ++s) {
      kf[s] = *reinterpret_cast<const half8_t*>(kp + 16 * s);
      vf[s] = *reinterpret_cast<const half8_t*>(vp + 16 * s);
    }
  }
  const int qstart = k0;  // causal: rows below k0 see no key here (k0 is a multiple of 64)
  const int n_qt = (len - qstart + kRowsT - 1) / kRowsT;
  const uint16_t* qbase = a.q + static_cast<int64_t>(s0) * a.q_tok + head * a.q_head;
  const uint16_t* dbase = a.dout + static_cast<int64_t>(s0) * a.do_tok + head * a.do_head;
  const __amdgpu_buffer_rsrc_t lrs = __builtin_amdgcn_make_buffer_rsrc(
      a.lse2 + static_cast<int64_t>(head) * a.n_tokens + s0, 0, len * 4, 0x00020000);
  const __amdgpu_buffer_rsrc_t drs = __builtin_amdgcn_make_buffer_rsrc(
      a.dd + static_cast<int64_t>(head) * a.n_tokens + s0, 0, len * 4, 0x00020000);
  TileDma qd, od;
  qd.init(a.q_tok, wave, lane);
  od.init(a.do_tok, wave, lane);
  auto issue = [&](int qt, int slot) __attribute__((always_inline)) {
    unsigned char* dst = smem + slot * kBwdSlot;
    const int r0 = qstart + qt * kRowsT;
    qd.issue(qbase + static_cast<int64_t>(r0) * a.q_tok, len - r0, dst, wave);
    od.issue(dbase + static_cast<int64_t>(r0) * a.do_tok, len - r0, dst + kTileBytes, wave);
    // the tile's 64 lse and 64 Dd values, one 4-byte load per lane (rows past len read 0), into
    // this wavefront's own copy (read by it alone)
    const uint32_t off = static_cast<uint32_t>((r0 + lane) * 4);
    unsigned char* st = dst + 2 * kTileBytes + wave * 512;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(lrs, (lds_ptr_t)(st), 4, off, 0, 0, 0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(drs, (lds_ptr_t)(st + 256), 4, off, 0, 0, 0);
  };

  BwdReads rd;
  rd.init(lds_addr(smem), lane);
  uint32_t lrow = lds_addr(smem) + 2 * kTileBytes + wave * 512 + 16 * hh;  // the rows' lse; Dd 256 on
  f32x16 dka[kD / 32], dva[kD / 32], sc, dp;  // sc, dp: the scores and dP of the block in hand
#pragma unroll
  for (int j = 0; j < kD / 32; ++j)
#pragma unroll
    for (int v = 0; v < 16; ++v) dka[j][v] = dva[j][v] = 0.f;
  half8_t pb[2][2], sb[2][2];  // [block][16-row group]: P and dS, packed
  f32x4_t l4[4], d4[4];        // the block's rows' lse and Dd
  half4_t tr[16];              // transposed operands of a 16-row group: [column block][dO, Q][halves]
  // P and dS of value v of the block (row 8 (v / 4) + 4 hh + v % 4 of it)
  auto value = [&](int blk, int v) __attribute__((always_inline)) {
    const float p = exp2_(__builtin_fmaf(sc[v], a.scale_log2, -l4[v >> 2][v & 3]));
    pb[blk][v >> 3][v & 7] = static_cast<_Float16>(p);
    sb[blk][v >> 3][v & 7] = static_cast<_Float16>(p * (dp[v] - d4[v >> 2][v & 3]));
  };
  // ... 0 where masked, for the block whose first row is q0 (query row < key or past the sequence,
  // key past the sequence): only where some row is masked for some key of the wavefront, a uniform
  // branch that holds no MFMA (with two copies of the products the accumulators were moved)
  auto mask = [&](int blk, int q0) __attribute__((always_inline)) {
    if (q0 < wk0 + 31 || q0 + 32 > len || wk0 + 32 > len) {
      int lo = key - q0 - 4 * hh;
      const int hi = q_end - q0 - 4 * hh;
      asm volatile("" : "+v"(lo));  // a real branch: selects on lo cannot be hoisted out of it
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int r = 8 * (v >> 2) + (v & 3);
        const bool in = r >= lo && r < hi;
        pb[blk][v >> 3][v & 7] = in ? pb[blk][v >> 3][v & 7] : static_cast<_Float16>(0.f);
        sb[blk][v >> 3][v & 7] = in ? sb[blk][v >> 3][v & 7] : static_cast<_Float16>(0.f);
      }
    }
  };
  // operand i (column block i / 2, dO or Q) of 16-row group g of block kB
  auto read_t = [&](auto blk, int g, int i) __attribute__((always_inline)) {
    constexpr int kB = decltype(blk)::value;
    const int off = kB * 8192 + g * 4096 + (i & 1 ? 0 : kTileBytes);
    tr[2 * i] = read_tr_untracked(rd.tlo[i >> 1], off);
    tr[2 * i + 1] = read_tr_untracked(rd.thi[i >> 1], off);
  };
  // block kB of the tile at the row addresses: S and dP, its lse and Dd, and (kPrev) the first group
  // of the transposed operands of the block before it
  auto scores = [&](auto blk, auto prev) __attribute__((always_inline)) {
    constexpr int kB = decltype(blk)::value;
    constexpr bool kPrev = decltype(prev)::value;
    half8_t f[8];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      f[2 * s] = read16_untracked(rd.row[s], kB * 8192);
      f[2 * s + 1] = read16_untracked(rd.row[s], kTileBytes + kB * 8192);
    }
#pragma unroll
    for (int g = 0; g < 4; ++g) l4[g] = read_f4_untracked(lrow, kB * 128 + g * 32);
#pragma unroll
    for (int g = 0; g < 4; ++g) d4[g] = read_f4_untracked(lrow, 256 + kB * 128 + g * 32);
#pragma unroll
    for (int v = 0; v < 16; ++v) sc[v] = dp[v] = 0.f;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const int x = 2 * (s & 3);
      // outstanding behind the operands: s < 4: the other row reads and the 8 lse / Dd reads, 14
      // behind the pair (15, the field's largest value, would be no wait); then the other row
      // reads and, from s = 5 on, 4 transposed reads per step
      if (s < 4) lgkm_wait(14, f[x], f[x + 1]);
      else lgkm_wait((7 - 2 * (s - 4)) + (kPrev ? 4 * (s - 4) : 0), f[x]);
      sc = __builtin_amdgcn_mfma_f32_32x32x16_f16(f[x], kf[s], sc, 0, 0, 0);
      if (s >= 4) lgkm_wait((6 - 2 * (s - 4)) + (kPrev ? 4 * (s - 4) : 0), f[x + 1]);
      dp = __builtin_amdgcn_mfma_f32_32x32x16_f16(f[x + 1], vf[s], dp, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if (s < 4) {
        f[x] = read16_untracked(rd.row[s + 4], kB * 8192);
        f[x + 1] = read16_untracked(rd.row[s + 4], kTileBytes + kB * 8192);
      } else if constexpr (kPrev) {
        read_t(std::integral_constant<int, kB ^ 1>{}, 0, 2 * (s - 4));
        read_t(std::integral_constant<int, kB ^ 1>{}, 0, 2 * (s - 4) + 1);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    // the lse / Dd reads have returned (they were issued before the second row reads)
    lgkm_landed(l4);
    lgkm_landed(d4);
  };
  // dV^T[d][key] += dO^T[d][q] P[q][key], dK^T[d][key] += Q^T[d][q] dS[q][key] of block kB (its first
  // group's operands in flight); beside each MFMA (kNext) a value of the other block
  auto gather = [&](auto blk, auto next) __attribute__((always_inline)) {
    constexpr int kB = decltype(blk)::value;
    constexpr bool kNext = decltype(next)::value;
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      const int g = u >> 3, i = u & 7, j = i >> 1;
      lgkm_wait(g == 0 ? 14 : 14 - 2 * i, tr[2 * i], tr[2 * i + 1]);
      if (i & 1)
        dka[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(pair8(tr[2 * i], tr[2 * i + 1]), sb[kB][g], dka[j], 0, 0, 0);
      else
        dva[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(pair8(tr[2 * i], tr[2 * i + 1]), pb[kB][g], dva[j], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if (g == 0) read_t(blk, 1, i);
      if constexpr (kNext) value(kB ^ 1, u);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  using B0 = std::integral_constant<int, 0>;
  using B1 = std::integral_constant<int, 1>;
  const int t0 = (wk0 - qstart) / kRowsT;  // the first tile with a row at or past the wavefront's keys
  int slot = 0;  // of the tile in hand
  issue(0, 0);
  auto arrive = [&](int t) __attribute__((always_inline)) {
    wait_vmcnt<0>();
    lds_barrier();  // tile t has landed; everyone is done with tile t - 2, whose slot takes t + 1
    if (t + 1 < n_qt) issue(t + 1, slot == 2 ? 0 : slot + 1);
  };
  auto leave = [&]() __attribute__((always_inline)) {
    rd.next_row(slot_step(slot));
    lrow += slot_step(slot);
    slot = slot == 2 ? 0 : slot + 1;
  };
  for (int t = 0; t < t0 && t < n_qt; ++t) {
    arrive(t);
    rd.next_t(slot_step(slot));
    leave();
  }
  if (t0 < n_qt) {
    const int q0 = qstart + t0 * kRowsT;
    arrive(t0);
    scores(B0{}, std::false_type{});
#pragma unroll
    for (int v = 0; v < 16; ++v) value(0, v);
    mask(0, q0);
    scores(B1{}, std::true_type{});
    gather(B0{}, std::true_type{});
    mask(1, q0 + 32);
    leave();
    for (int t = t0 + 1; t < n_qt; ++t) {
      const int r0 = qstart + t * kRowsT;
      arrive(t);
      scores(B0{}, std::true_type{});
      gather(B1{}, std::true_type{});
      mask(0, r0);
      rd.next_t(slot_step(slot == 0 ? 2 : slot - 1));
      scores(B1{}, std::true_type{});
      gather(B0{}, std::true_type{});
      mask(1, r0 + 32);
      leave();
    }
    // the last block: nothing to run beside it (as in dQ: no read is in flight)
    asm volatile("s_waitcnt lgkmcnt(0)");
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 8; ++i) read_t(B1{}, 0, i);
    gather(B1{}, std::false_type{});
  }
  // fp32 partials [head][token][d]. A lane holds its key's column of the accumulators (rows
  // d = 32 j + 8 (v / 4) + 4 hh + v % 4): stored as they are, every store instruction would touch
  // 64 rows 16 bytes each. Each wavefront stages its 32 keys x 128 columns in its own part of the
  // ring instead (rows of 132 floats: the 16 lanes of a write phase meet 16 distinct bank groups)
  // and stores whole rows, two per instruction.
  done();
  __syncthreads();  // every wavefront is done with the ring
  constexpr int kStageLd = kD + 4;
  float* stage = reinterpret_cast<float*>(smem) + wave * 32 * kStageLd;
  auto store_rows = [&](const f32x16 (&acc)[kD / 32], float mul, float* part) {
#pragma unroll
    for (int j = 0; j < kD / 32; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<float4*>(&stage[l32 * kStageLd + 32 * j + 8 * g + 4 * hh]) =
            make_float4(acc[j][4 * g] * mul, acc[j][4 * g + 1] * mul, acc[j][4 * g + 2] * mul,
                        acc[j][4 * g + 3] * mul);
    // the wavefront reads back its own rows: its LDS writes complete first
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    u32x4 x[16];
#pragma unroll
    for (int it = 0; it < 16; ++it) {
      const int r = 2 * it + (lane >> 5), c = lane & 31;
      x[it] = *reinterpret_cast<const u32x4*>(&stage[r * kStageLd + 4 * c]);
    }
    const __amdgpu_buffer_rsrc_t prs =
        store_rsrc(part + (static_cast<int64_t>(head) * a.n_tokens + s0 + wk0) * kD);
#pragma unroll
    for (int it = 0; it < 16; ++it) {
      const int r = 2 * it + (lane >> 5), c = lane & 31;
      store16(prs, wk0 + r < len ? static_cast<uint32_t>((r * kD + 4 * c) * 4) : kOob, x[it]);
    }
    // the next call overwrites the rows: every read above has returned first
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  };
  store_rows(dka, a.scale, a.dk_part);
  store_rows(dva, 1.f, a.dv_part);
}

// dQ and the dK / dV partials in one launch: they read the same inputs and write disjoint
// outputs, and each alone has fewer workgroups than the chip has CUs (its time is its longest
// workgroup's), so side by side they share the chip. The grid is (query head, sequence,
// 2 x rank): every sequence's longest work is dispatched first, rank by rank, so the workgroups
// that wait for a free CU are the shortest ones. Rank r of a sequence of n tiles is dQ query tile
// n - 1 - r (even z) and dK / dV key tile r (odd z); ranks past n exit at once.
template <int W>
__global__ __launch_bounds__(64 * W, 1) void attn_bwd_kernel(BwdArgs a) {
  __shared__ __attribute__((aligned(1024))) unsigned char smem[kBwdLds];
  const int rank = static_cast<int>(blockIdx.z) >> 1;
  const int len = a.cu[blockIdx.y + 1] - a.cu[blockIdx.y];
  const int n_own = (len + 32 * W - 1) / (32 * W);
  if (rank >= n_own) return;  // the whole workgroup, before any barrier
  if ((blockIdx.z & 1) == 0)
    attn_bwd_dq<W>(a, blockIdx.y, blockIdx.x, n_own - 1 - rank, smem, [] {});
  else
    attn_bwd_dkdv<W>(a, blockIdx.y, blockIdx.x, rank, smem, [] {});
}

// The same work from a queue: one workgroup per CU takes items until none is left, the longest
// first. With one workgroup per item the dispatcher deals them round-robin over XCDs and shader
// engines whatever their lengths, and in order, so that a full engine holds back the others: of
// the launch's 511 us at lengths [4096, 3001, 2222, 1531] (12 / 2 heads) a CU worked 377, of 76 us
// at 16 rows of 128..512 tokens 51. Backward (all launches): 538 -> 463 us and 94.6 -> 82.
//
// An item is a (sequence, 128-token tile, dK/dV or dQ, head); its length follows the sequence's
// tiles from there on (dK / dV: the query tiles after its keys; dQ: the key tiles before its
// rows), the m of list_pair.
template <int W>
__global__ __launch_bounds__(64 * W, 1) void attn_bwd_queue_kernel(BwdArgs a) {
  // the next item's index behind the ring
  __shared__ __attribute__((aligned(1024))) unsigned char smem[kBwdLds + 16];
  const int lane = threadIdx.x & 63;
  const int len = lane < a.n_seqs ? a.cu[lane + 1] - a.cu[lane] : 0;
  const int own = min((max(len, 0) + 32 * W - 1) / (32 * W), a.n_tiles);
  const unsigned pairs = static_cast<unsigned>(wave_count(own));
  const unsigned per_pair = 2u * static_cast<unsigned>(a.n_q_heads);
  unsigned item = blockIdx.x;
  for (;;) {
    const unsigned pair = item / per_pair;
    if (pair >= pairs) break;
    int seq;
    const int lo = list_pair(own, a.n_tiles, pair, lane, seq);
    const int rank = __builtin_amdgcn_readlane(own, seq) - lo;
    const int which = static_cast<int>(item - pair * per_pair);
    // the next item is drawn when this one's products are done, while its results go out (drawn
    // before, the longest items would each hold back one more)
    unsigned next = 0xffffffffu;  // past every item
    auto draw = [&]() __attribute__((always_inline)) {
      if (threadIdx.x == 0) next = atomicAdd(a.counter, 1u);
    };
    if (which < a.n_q_heads)
      attn_bwd_dkdv<W>(a, seq, which, rank, smem, draw);
    else
      attn_bwd_dq<W>(a, seq, which - a.n_q_heads, lo - 1, smem, draw);
    // the next item's counted waits start from nothing in flight, its ring from idle slots
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) *reinterpret_cast<unsigned*>(smem + kBwdLds) = next;
    __syncthreads();
    item = __builtin_amdgcn_readfirstlane(*reinterpret_cast<const unsigned*>(smem + kBwdLds));
  }
}

// dK / dV fp16 [token][kv head][d] = sum over the KV head's query heads, in head order. A
// thread takes 4 columns d and, with the rotary backward (a.cos), also their partners d + 64:
// dK's pairs are rotated back in fp32 before the rounding.
// dK / dV partials of the KV head's query heads at columns d_c .. d_c + 3 (c < C), summed in head
// order; every load of eight heads is in flight before their adds.
template <int C>
__device__ __forceinline__ void sum_heads4(const BwdArgs& a, int kvh, int64_t t, const int (&d)[C],
                                           float (&k)[C][4], float (&v)[C][4]) {
#pragma unroll
  for (int c = 0; c < C; ++c)
#pragma unroll
    for (int e = 0; e < 4; ++e) k[c][e] = v[c][e] = 0.f;
  const int64_t head_stride = a.n_tokens * kD;
  const int64_t off0 = (static_cast<int64_t>(kvh) * a.group * a.n_tokens + t) * kD;
  for (int g0 = 0; g0 < a.group; g0 += 8) {
    float4 xk[8][C], xv[8][C];
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const int64_t off = off0 + (g0 + j < a.group ? g0 + j : 0) * head_stride + d[c];
        xk[j][c] = *reinterpret_cast<const float4*>(a.dk_part + off);
        xv[j][c] = *reinterpret_cast<const float4*>(a.dv_part + off);
      }
    // selects, not a branch: a branch between the loads and the adds would let the compiler sink
    // each load to its add, one round trip per head (heads past the group add +0)
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const bool in = g0 + j < a.group;
#pragma unroll
      for (int c = 0; c < C; ++c) {
        k[c][0] += in ? xk[j][c].x : 0.f; k[c][1] += in ? xk[j][c].y : 0.f;
        k[c][2] += in ? xk[j][c].z : 0.f; k[c][3] += in ? xk[j][c].w : 0.f;
        v[c][0] += in ? xv[j][c].x : 0.f; v[c][1] += in ? xv[j][c].y : 0.f;
        v[c][2] += in ? xv[j][c].z : 0.f; v[c][3] += in ? xv[j][c].w : 0.f;
      }
    }
  }
}

template <bool kRope>
__global__ __launch_bounds__(256) void attn_bwd_reduce_kernel(BwdArgs a) {
  constexpr int kGroups = kRope ? kD / 8 : kD / 4;  // threads per (token, KV head)
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const int64_t total = a.n_tokens * a.n_kv_heads * kGroups;
  if (idx >= total) return;
  const int c4 = static_cast<int>(idx % kGroups);
  const int64_t tk = idx / kGroups;
  const int kvh = static_cast<int>(tk % a.n_kv_heads);
  const int64_t t = tk / a.n_kv_heads;
  uint16_t* dk = a.dk + t * a.dk_tok + kvh * a.dk_head;
  uint16_t* dv = a.dv + t * a.dv_tok + kvh * a.dv_head;
  constexpr int C = kRope ? 2 : 1;  // with the rotary backward: the (d, d + 64) column pairs
  int d[C];
  d[0] = 4 * c4;
  if constexpr (kRope) d[C - 1] = 4 * c4 + kD / 2;
  float kk[C][4], vv[C][4];
  sum_heads4<C>(a, kvh, t, d, kk, vv);
  float(&k1)[4] = kk[0];
  float(&v1)[4] = vv[0];
  if constexpr (kRope) {
    float(&k2)[4] = kk[C - 1];
    float(&v2)[4] = vv[C - 1];
    rope_back4(k1, k2, a.cos + t * a.cs_tok, a.sin + t * a.cs_tok, 4 * c4);
    *reinterpret_cast<uint2*>(dk + 4 * c4 + kD / 2) = make_uint2(pack2(k2[0], k2[1]), pack2(k2[2], k2[3]));
    *reinterpret_cast<uint2*>(dv + 4 * c4 + kD / 2) = make_uint2(pack2(v2[0], v2[1]), pack2(v2[2], v2[3]));
  }
  *reinterpret_cast<uint2*>(dk + 4 * c4) = make_uint2(pack2(k1[0], k1[1]), pack2(k1[2], k1[3]));
  *reinterpret_cast<uint2*>(dv + 4 * c4) = make_uint2(pack2(v1[0], v1[1]), pack2(v1[2], v1[3]));
}

}  // namespace
}  // namespace talm

using namespace talm;

TALM_API int talm_attn_fwd(const uint16_t* q, int64_t q_stride_tok, int64_t q_stride_head,
                           const uint16_t* k, int64_t k_stride_tok, int64_t k_stride_head,
                           const uint16_t* v, int64_t v_stride_tok, int64_t v_stride_head,
                           const int32_t* cu_seqlens, int32_t n_seqs, int32_t max_seqlen,
                           int64_t n_tokens, int32_t n_q_heads, int32_t n_kv_heads,
                           int32_t head_dim, float scale, uint16_t* out, int64_t o_stride_tok,
                           int64_t o_stride_head, float* lse, void* stream) {
  if (head_dim != kD)
    return fail(TALM_EINVAL, "attn_fwd: head_dim %d (only %d)", head_dim, kD);
  if (n_seqs < 0 || max_seqlen < 0 || n_tokens < 0 || n_q_heads < 1 || n_kv_heads < 1 ||
      n_q_heads % n_kv_heads || n_tokens >= (int64_t{1} << 31))
    return fail(TALM_EINVAL, "attn_fwd: bad shape (seqs %d, max_seqlen %d, tokens %lld, heads %d/%d)",
                n_seqs, max_seqlen, (long long)n_tokens, n_q_heads, n_kv_heads);
  for (int64_t s : {q_stride_tok, q_stride_head, k_stride_tok, k_stride_head, v_stride_tok,
                    v_stride_head, o_stride_tok, o_stride_head})
    if (s < 0 || s % 8)
      return fail(TALM_EINVAL, "attn_fwd: strides must be non-negative multiples of 8 elements");
  if (k_stride_tok >= (int64_t{1} << 23) || v_stride_tok >= (int64_t{1} << 23) ||
      o_stride_tok >= (int64_t{1} << 23))
    return fail(TALM_EINVAL, "attn_fwd: k / v / out token strides must be below 2^23 elements");
  if (n_seqs == 0 || max_seqlen == 0 || n_tokens == 0) return ok();
  if (!q || !k || !v || !cu_seqlens || !out || !lse) return fail(TALM_EINVAL, "attn_fwd: null pointer");
  if (!aligned(q, 16) || !aligned(k, 16) || !aligned(v, 16) || !aligned(out, 16))
    return fail(TALM_EINVAL, "attn_fwd: q, k, v and out must be 16-byte aligned");
  const int group = n_q_heads / n_kv_heads;
  // query heads per workgroup (4 wavefronts): 4, 2 or 1, what divides the group; three with an idle
  // wavefront where a group is a multiple of three and no sequence has more than 64 rows, of which
  // one head would keep at most two wavefronts busy (12 heads on 4 KV heads, one head / three: 256
  // rows of 16 tokens 26.8 / 12.9 us, 64 of 33 10.0 / 7.8, 65 of 64 14.6 / 12.9)
  const bool three = group % 3 == 0 && group % 2 != 0 && max_seqlen <= 64;
  const int h = three || group % 4 == 0 ? 4 : group % 2 == 0 ? 2 : 1;
  const int rows = 32 * (4 / h), wg_heads = three ? 3 : h;
  FwdArgs a{};
  a.q = q; a.q_tok = q_stride_tok; a.q_head = q_stride_head;
  a.k = k; a.k_tok = k_stride_tok; a.k_head = k_stride_head;
  a.v = v; a.v_tok = v_stride_tok; a.v_head = v_stride_head;
  a.cu = cu_seqlens; a.group = group; a.wg_heads = wg_heads;
  a.head_chunks = group / wg_heads;
  a.scale_log2 = scale * 1.44269504088896341f;
  a.out = out; a.o_tok = o_stride_tok; a.o_head = o_stride_head;
  a.lse = lse; a.n_tokens = n_tokens;
  // rank-major, so that every sequence's longest workgroups start first; more ranks than a grid's
  // third axis holds go on its first one
  const unsigned chunks = static_cast<unsigned>(n_q_heads / wg_heads), seqs = static_cast<unsigned>(n_seqs);
  const unsigned ranks = static_cast<unsigned>((static_cast<int64_t>(max_seqlen) + rows - 1) / rows);
  a.rank_x = ranks > 65535;
  dim3 grid = a.rank_x ? dim3(ranks, chunks, seqs) : dim3(chunks, seqs, ranks);
  // Split the key tiles (S = 2) where the longest workgroup's chain, not the chip, sets the time:
  // the workgroups (estimated: the lengths are on the device) fit one round, one per CU, and the
  // chain is at least 8 tiles; or they fit two rounds and the chain is long enough (16 tiles) to
  // pay for the second one. Measured, S = 1 / 2, 12 query heads on 2 KV heads: lengths [2048] 38.8 /
  // 32.7 us, [4096] 79.7 / 66.8, [900, 700, 333] 21.0 / 18.5; [300, 211] 9.3 / 9.9; 8 rows of
  // 128..512 15.2 / 17.7, 8 of 1024 39.4 / 47.1, [4096, 3001, 2222, 1531] 132 / 139.
  const int64_t wgs = (n_tokens + static_cast<int64_t>(n_seqs) * rows / 2) / rows * chunks;
  const int64_t cus = device_cus(), chain = (static_cast<int64_t>(max_seqlen) + kKeys - 1) / kKeys;
  const bool split = wgs <= cus ? chain >= 8 : wgs <= 2 * cus && chain >= 16;
  // Workgroups by list_pair's list, longest first over all sequences, where they exceed a round (two
  // per CU) and the sequences differ in length (an eighth of the rectangle empty): round-robin over
  // XCDs by sequence, the longest sequences' workgroups meet on some of them. Grid / list: 16 rows of
  // 1..1024 40.8 / 34.9 us, [4096, 3001, 2222, 1531] 135 / 120; but eight of 1024 38.7 / 40.8 and of
  // 2048 119 / 121.5, 16 rows of 128..512 (one round) 19.0 / 20.0: finding a tile costs about 0.5 us.
  const int64_t items = std::min<int64_t>(n_tokens / rows + n_seqs, static_cast<int64_t>(n_seqs) * ranks) * chunks;
  if (n_seqs <= kListSeqs && wgs > 2 * cus && 8 * n_tokens < 7 * static_cast<int64_t>(n_seqs) * max_seqlen &&
      items < (int64_t{1} << 30)) {
    a.n_seqs = n_seqs;
    a.chunks = chunks;
    a.list_tiles = static_cast<int>(ranks);
    grid = dim3(static_cast<unsigned>(items));
  }
  const hipStream_t s = as_stream(stream);
#define TALM_ATTN_FWD(H)                                                                         \
  if (split)                                                                                     \
    hipLaunchKernelGGL((attn_fwd_kernel<H, 2>), grid, dim3(512), 0, s, a);                       \
  else                                                                                           \
    hipLaunchKernelGGL((attn_fwd_kernel<H, 1>), grid, dim3(256), 0, s, a)
  if (h == 4) { TALM_ATTN_FWD(4); }
  else if (h == 2) { TALM_ATTN_FWD(2); }
  else { TALM_ATTN_FWD(1); }
#undef TALM_ATTN_FWD
  return check_launch("attn_fwd");
}

static constexpr int64_t kQueueBytes = 256;  // the work queue's counter, at the workspace's end

TALM_API int64_t talm_attn_bwd_workspace(int64_t n_tokens, int32_t n_q_heads) {
  if (n_tokens < 0 || n_q_heads < 1) return -1;
  // Dd and lse2 [Hq, N] f32, then the dK and dV partials [Hq, N, D] f32 each (256-byte aligned
  // parts)
  const int64_t dd = (n_tokens * n_q_heads * 4 + 255) / 256 * 256;
  return 2 * dd + 2 * n_tokens * n_q_heads * kD * 4 + kQueueBytes;
}

namespace talm {
namespace {

int attn_bwd_impl(const uint16_t* q, int64_t q_stride_tok, int64_t q_stride_head,
                  const uint16_t* k, int64_t k_stride_tok, int64_t k_stride_head,
                  const uint16_t* v, int64_t v_stride_tok, int64_t v_stride_head,
                  const uint16_t* out, int64_t o_stride_tok, int64_t o_stride_head,
                  const uint16_t* dout, int64_t do_stride_tok, int64_t do_stride_head,
                  const float* lse, const int32_t* cu_seqlens, int32_t n_seqs,
                  int32_t max_seqlen, int64_t n_tokens, int32_t n_q_heads, int32_t n_kv_heads,
                  int32_t head_dim, float scale, const float* cos, const float* sin,
                  int64_t cs_stride, uint16_t* dq, int64_t dq_stride_tok,
                  int64_t dq_stride_head, uint16_t* dk, int64_t dk_stride_tok,
                  int64_t dk_stride_head, uint16_t* dv, int64_t dv_stride_tok,
                  int64_t dv_stride_head, void* workspace, int64_t workspace_bytes,
                  void* stream) {
  if (head_dim != kD)
    return fail(TALM_EINVAL, "attn_bwd: head_dim %d (only %d)", head_dim, kD);
  if (n_seqs < 0 || max_seqlen < 0 || n_tokens < 0 || n_q_heads < 1 || n_kv_heads < 1 ||
      n_q_heads % n_kv_heads || n_tokens >= (int64_t{1} << 31))
    return fail(TALM_EINVAL, "attn_bwd: bad shape (seqs %d, max_seqlen %d, tokens %lld, heads %d/%d)",
                n_seqs, max_seqlen, (long long)n_tokens, n_q_heads, n_kv_heads);
  for (int64_t s : {q_stride_tok, q_stride_head, k_stride_tok, k_stride_head, v_stride_tok,
                    v_stride_head, o_stride_tok, o_stride_head, do_stride_tok, do_stride_head,
                    dq_stride_tok, dq_stride_head, dk_stride_tok, dk_stride_head, dv_stride_tok,
                    dv_stride_head})
    if (s < 0 || s % 8)
      return fail(TALM_EINVAL, "attn_bwd: strides must be non-negative multiples of 8 elements");
  if (q_stride_tok >= (int64_t{1} << 23) || k_stride_tok >= (int64_t{1} << 23) ||
      v_stride_tok >= (int64_t{1} << 23) || do_stride_tok >= (int64_t{1} << 23) ||
      dq_stride_tok >= (int64_t{1} << 23))
    return fail(TALM_EINVAL, "attn_bwd: q / k / v / dout / dq token strides must be below 2^23 elements");
  if (n_seqs > 65535 || (max_seqlen + 127) / 128 > 32767)
    return fail(TALM_EINVAL, "attn_bwd: at most 65535 sequences of at most 4194176 tokens");
  // (a workspace without the queue's counter is accepted: one workgroup per item then)
  const int64_t need = talm_attn_bwd_workspace(n_tokens, n_q_heads) - kQueueBytes;
  if (workspace_bytes < need)
    return fail(TALM_EINVAL, "attn_bwd: workspace of %lld bytes, %lld needed",
                (long long)workspace_bytes, (long long)need);
  const bool rope = cos != nullptr || sin != nullptr;
  if (rope && (cs_stride < kD || cs_stride % 4 || cs_stride >= (int64_t{1} << 24)))
    return fail(TALM_EINVAL, "attn_bwd: cos / sin row stride %lld (at least %d, a multiple of 4)",
                (long long)cs_stride, kD);
  if (n_seqs == 0 || max_seqlen == 0 || n_tokens == 0) return ok();
  if (!q || !k || !v || !out || !dout || !lse || !cu_seqlens || !dq || !dk || !dv || !workspace)
    return fail(TALM_EINVAL, "attn_bwd: null pointer");
  if (rope && (!cos || !sin || !aligned(cos, 16) || !aligned(sin, 16)))
    return fail(TALM_EINVAL, "attn_bwd: cos and sin both given, 16-byte aligned");
  if (!aligned(q, 16) || !aligned(k, 16) || !aligned(v, 16) || !aligned(out, 16) ||
      !aligned(dout, 16) || !aligned(dq, 16) || !aligned(dk, 8) || !aligned(dv, 8) ||
      !aligned(workspace, 256))
    return fail(TALM_EINVAL, "attn_bwd: operands 16-byte aligned (dk, dv 8), workspace 256");
  constexpr int W = 4;
  BwdArgs a{};
  a.q = q; a.q_tok = q_stride_tok; a.q_head = q_stride_head;
  a.k = k; a.k_tok = k_stride_tok; a.k_head = k_stride_head;
  a.v = v; a.v_tok = v_stride_tok; a.v_head = v_stride_head;
  a.o = out; a.o_tok = o_stride_tok; a.o_head = o_stride_head;
  a.dout = dout; a.do_tok = do_stride_tok; a.do_head = do_stride_head;
  a.lse = lse; a.cu = cu_seqlens;
  a.group = n_q_heads / n_kv_heads; a.n_q_heads = n_q_heads; a.n_kv_heads = n_kv_heads;
  a.n_tiles = (max_seqlen + 32 * W - 1) / (32 * W);
  a.scale = scale; a.scale_log2 = scale * 1.44269504088896341f;
  a.n_tokens = n_tokens;
  unsigned char* ws = static_cast<unsigned char*>(workspace);
  const int64_t dd_bytes = (n_tokens * n_q_heads * 4 + 255) / 256 * 256;
  a.dd = reinterpret_cast<float*>(ws);
  a.lse2 = reinterpret_cast<float*>(ws + dd_bytes);
  a.dk_part = reinterpret_cast<float*>(ws + 2 * dd_bytes);
  a.dv_part = a.dk_part + n_tokens * n_q_heads * kD;
  a.dq = dq; a.dq_tok = dq_stride_tok; a.dq_head = dq_stride_head;
  a.dk = dk; a.dk_tok = dk_stride_tok; a.dk_head = dk_stride_head;
  a.dv = dv; a.dv_tok = dv_stride_tok; a.dv_head = dv_stride_head;
  a.cos = rope ? cos : nullptr; a.sin = rope ? sin : nullptr; a.cs_tok = cs_stride;
  // The queue for more than two items per CU (what there is to balance), up to one sequence per lane,
  // where its indices fit 32 bits, and unless the items are all short (one tile per sequence, at most
  // 96 of its 128 rows on the average). Backward, grid / queue: [1500, 800] with 14 / 2 heads (532 items)
  // 78 / 72 us, eight rows of 128..512 (672) 59 / 51, [3000] (576) 137 / 134, but [2048] (384) 82.3
  // / 84.2, four rows of 128..512 (312) 34.9 / 35.9: finding and drawing an item costs 1-2 us. One
  // tile per sequence, 64 sequences of 33, 64, 96 and 128 tokens with 12 / 2 heads (1536): 46.3 / 52.8,
  // 60.2 / 61.3, 86.2 / 82.6, 105 / 94; 24 sequences, 16 / 16 heads (768): 31.9 / 35.0, 37.5 / 40.6,
  // 51.3 / 53.8, 60.5 / 60.6.
  const int64_t items = 2 * static_cast<int64_t>(n_q_heads) *
                        std::min<int64_t>(n_tokens / (32 * W) + n_seqs, static_cast<int64_t>(n_seqs) * a.n_tiles);
  a.n_seqs = n_seqs;
  if (n_seqs <= kListSeqs && items > 2 * device_cus() &&
      (a.n_tiles > 1 || n_tokens > 96 * static_cast<int64_t>(n_seqs)) && items < (int64_t{1} << 30) &&
      workspace_bytes >= need + kQueueBytes) {
    a.counter = reinterpret_cast<unsigned*>(a.dv_part + n_tokens * n_q_heads * kD);
    a.queue_wgs = static_cast<unsigned>(std::min<int64_t>(items, device_cus()));
  }
  const hipStream_t s = as_stream(stream);
  const int64_t rows = n_tokens * n_q_heads;
  hipLaunchKernelGGL(attn_bwd_dot_kernel, dim3(static_cast<unsigned>((rows * 16 + 255) / 256)),
                     dim3(256), 0, s, a);
  if (a.counter) {
    hipLaunchKernelGGL((attn_bwd_queue_kernel<W>), dim3(a.queue_wgs), dim3(64 * W), 0, s, a);
  } else {
    const dim3 grid(static_cast<unsigned>(n_q_heads), static_cast<unsigned>(n_seqs),
                    static_cast<unsigned>(2 * a.n_tiles));
    hipLaunchKernelGGL((attn_bwd_kernel<W>), grid, dim3(64 * W), 0, s, a);
  }
  const int64_t red = n_tokens * n_kv_heads * (rope ? kD / 8 : kD / 4);
  if (rope)
    hipLaunchKernelGGL(attn_bwd_reduce_kernel<true>, dim3(static_cast<unsigned>((red + 255) / 256)),
                       dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL(attn_bwd_reduce_kernel<false>, dim3(static_cast<unsigned>((red + 255) / 256)),
                       dim3(256), 0, s, a);
  return check_launch("attn_bwd");
}

}  // namespace
}  // namespace talm

TALM_API int talm_attn_bwd(const uint16_t* q, int64_t q_stride_tok, int64_t q_stride_head,
                           const uint16_t* k, int64_t k_stride_tok, int64_t k_stride_head,
                           const uint16_t* v, int64_t v_stride_tok, int64_t v_stride_head,
                           const uint16_t* out, int64_t o_stride_tok, int64_t o_stride_head,
                           const uint16_t* dout, int64_t do_stride_tok, int64_t do_stride_head,
                           const float* lse, const int32_t* cu_seqlens, int32_t n_seqs,
                           int32_t max_seqlen, int64_t n_tokens, int32_t n_q_heads,
                           int32_t n_kv_heads, int32_t head_dim, float scale, uint16_t* dq,
                           int64_t dq_stride_tok, int64_t dq_stride_head, uint16_t* dk,
                           int64_t dk_stride_tok, int64_t dk_stride_head, uint16_t* dv,
                           int64_t dv_stride_tok, int64_t dv_stride_head, void* workspace,
                           int64_t workspace_bytes, void* stream) {
  return attn_bwd_impl(q, q_stride_tok, q_stride_head, k, k_stride_tok, k_stride_head, v,
                       v_stride_tok, v_stride_head, out, o_stride_tok, o_stride_head, dout,
                       do_stride_tok, do_stride_head, lse, cu_seqlens, n_seqs, max_seqlen,
                       n_tokens, n_q_heads, n_kv_heads, head_dim, scale, nullptr, nullptr, 0, dq,
                       dq_stride_tok, dq_stride_head, dk, dk_stride_tok, dk_stride_head, dv,
                       dv_stride_tok, dv_stride_head, workspace, workspace_bytes, stream);
}

TALM_API int talm_attn_bwd_rope(const uint16_t* q, int64_t q_stride_tok, int64_t q_stride_head,
                                const uint16_t* k, int64_t k_stride_tok, int64_t k_stride_head,
                                const uint16_t* v, int64_t v_stride_tok, int64_t v_stride_head,
                                const uint16_t* out, int64_t o_stride_tok, int64_t o_stride_head,
                                const uint16_t* dout, int64_t do_stride_tok,
                                int64_t do_stride_head, const float* lse,
                                const int32_t* cu_seqlens, int32_t n_seqs, int32_t max_seqlen,
                                int64_t n_tokens, int32_t n_q_heads, int32_t n_kv_heads,
                                int32_t head_dim, float scale, const float* cos, const float* sin,
                                int64_t cs_stride, uint16_t* dq, int64_t dq_stride_tok,
                                int64_t dq_stride_head, uint16_t* dk, int64_t dk_stride_tok,
                                int64_t dk_stride_head, uint16_t* dv, int64_t dv_stride_tok,
                                int64_t dv_stride_head, void* workspace, int64_t workspace_bytes,
                                void* stream) {
  if (!cos || !sin) return fail(TALM_EINVAL, "attn_bwd_rope: cos and sin are required");
  return attn_bwd_impl(q, q_stride_tok, q_stride_head, k, k_stride_tok, k_stride_head, v,
                       v_stride_tok, v_stride_head, out, o_stride_tok, o_stride_head, dout,
                       do_stride_tok, do_stride_head, lse, cu_seqlens, n_seqs, max_seqlen,
                       n_tokens, n_q_heads, n_kv_heads, head_dim, scale, cos, sin, cs_stride, dq,
                       dq_stride_tok, dq_stride_head, dk, dk_stride_tok, dk_stride_head, dv,
                       dv_stride_tok, dv_stride_head, workspace, workspace_bytes, stream);
}

// Prompt-sized attention for gfx950 (MFMA 32x32x16 bf16): the query tiles of
// calls whose sequences bring many query rows (prefill, chunked prefill, the
// recomputation of a preempted sequence). Included by verify_attention.hip.
//
// A workgroup (4 waves) owns 128 query rows of one (sequence, kv head): the G
// query heads of consecutive tokens, as in the per-tile grid, 32 rows to a
// wave. The keys stream through LDS in steps of 64 that all waves share (the
// 16-row tiles of the other launches stream the whole context once for every
// 16 / G tokens), double-buffered: the next steps' rows are in flight into
// registers while this one is multiplied, and go to the other buffer after it
// (FP8 rows are decoded to bf16 there, once per workgroup instead of once per
// wave).
//   S^T[64 keys x 32 rows] = K (A operand, LDS) x Q^T (B operand, registers)
//   online softmax with the row on a lane pair (l, l + 32)
//   O^T[128 x 32 rows]    += V^T (A operand, transposing LDS reads) x P^T,
// P^T being the exponentiated S^T registers as they are: the 16-key chunk's
// k-slot (h, e) holds key 8 (e / 4) + 4h + e % 4 on both sides, so no lane
// exchange is needed.
//
// What bounds it: at 6301 tokens the SIMDs are at matrix work for 44% of the time
// and at vector work (the softmax, the stores of the next step) for 44%, the CUs'
// LDS at reads for 38%: two waves to a SIMD, in two workgroups, overlap the three
// that one wave does in turn. Short prompts are chains of steps on CUs half idle
// (ragged prompts up to 1021 tokens: 27% busy). 32 query heads over 8, one prompt,
// bf16, in 16-row tiles and here: 6301 tokens 1760 -> 375 us (185 -> 866 TFLOP/s),
// 1024 tokens 75 -> 30 us, four prompts of 512 84 -> 22 us. Measured and not kept:
// 64 rows per wave (half the LDS reads, but one wave per SIMD: 452 us), the next
// step's scores beside this step's softmax in one wave (400 us), eight waves in two
// groups half a step apart (369 us at 6301 tokens, 34 us at 1024).
#pragma once

namespace hs {

typedef float f32x16_t __attribute__((ext_vector_type(16)));

constexpr int kPfStep = 64;              // keys per step
constexpr int kPfWaves = 4;
constexpr int kPfTileRows = kPfWaves * 32;  // query rows per workgroup
constexpr int kPfAhead = 12;             // LDS reads issued ahead of the matrix work
constexpr int kPfTileB = kPfStep * 256;  // bytes of one K or V tile (bf16 rows)

// 16-byte chunk c of tile row kk is stored at chunk c ^ pf_swz(kk): the K
// operand reads (16 consecutive rows at one chunk) and the V transposing reads
// (rows 4h .. 4h + 3 at four adjacent chunks) then touch every bank once.
__device__ __forceinline__ int pf_swz(int kk) { return ((kk & 3) << 2) | ((kk >> 2) & 3); }

// A thread's share of one step's K and V rows on their way from the cache to
// LDS: piece i is 16 bytes of row kk(i).
template <bool kFp8>
struct PfStage {
  static constexpr int kLanesPerRow = (kFp8 ? 128 : 256) / 16;
  static constexpr int kRowsPerPiece = kPfWaves * 64 / kLanesPerRow;
  static constexpr int kRowsPerWave = 64 / kLanesPerRow;
  static constexpr int kPieces = kPfStep / kRowsPerPiece;
};

// Where the sequence's key rows are. Blocks hold a power of two of tokens, at
// least 32, so a 32-key half of a step lies in one block; the block-table
// entries [base, base + 64) sit in the lanes of one register (lane j: entry
// base + j), so a lookup is a v_readlane. Unpaged rows are one endless block.
struct PfTable {
  int shift, nbt, base, entry;
  int64_t s_blk;
};

// block-table entry i of sequence b: -1 for what is no block of the cache
__device__ __forceinline__ int pf_entry(const AttnArgs& a, int b, int i, int nbt) {
  if (a.contig) return 0;
  if (i >= nbt || i >= a.bt_width) return -1;
  const int e = a.bt[(int64_t)b * a.bt_stride + i];
  return e < a.num_blocks ? e : -1;
}

// Element offsets of the two 32-key halves of step i, and the clamp of its
// rows: lim is the last visible key's row of the step (63 or more: all rows
// are visible); a half past it reads the first half instead. Steps from T on
// (the end of the workgroup's steps) read the last one again.
struct PfStep {
  int64_t off[2];
  int lim;
};

__device__ __forceinline__ PfStep pf_step(const AttnArgs& a, int b, int i, int T, int khi,
                                          PfTable& tab) {
  PfStep s;
  i = i < T ? i : T - 1;
  const int ws = i * kPfStep;
  s.lim = khi - 1 - ws;
  const int e0 = ws >> tab.shift;
  if (e0 >= tab.base + 64) {  // a step's entries never straddle a group of 64
    tab.base = e0 & ~63;
    tab.entry = pf_entry(a, b, tab.base + (threadIdx.x & 63), tab.nbt);
  }
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int key = (h && s.lim >= 32) ? ws + 32 : ws;
    const int e = key >> tab.shift;
    const int blk = __builtin_amdgcn_readlane(tab.entry, e - tab.base);
    s.off[h] = (int64_t)(blk > 0 ? blk : 0) * tab.s_blk +
               (int64_t)(key - (e << tab.shift)) * a.c_st;
  }
  return s;
}

// a thread's pieces of one step's rows of one cache (K or V; `cache` at the
// kv head, and at the sequence's first row where unpaged)
template <bool kFp8>
__device__ __forceinline__ void pf_load(const uint8_t* cache, const PfStep& s, uint32_t rowb,
                                        int wid, uint4 (&x)[PfStage<kFp8>::kPieces]) {
  using S = PfStage<kFp8>;
  const int lane = threadIdx.x & 63;
  const int row = lane / S::kLanesPerRow, sub = lane % S::kLanesPerRow;
#pragma unroll
  for (int i = 0; i < S::kPieces; ++i) {
    const int r0 = i * S::kRowsPerPiece + wid * S::kRowsPerWave;  // the wave's first row
    const int h = r0 >> 5;
    const int lim = (h && s.lim >= 32) ? s.lim - 32 : s.lim;
    const int r = min((r0 & 31) + row, lim);
    const uint8_t* base = cache + (h ? s.off[1] : s.off[0]) * (kFp8 ? 1 : 2);
    x[i] = *reinterpret_cast<const uint4*>(base + ((uint32_t)r * rowb + sub * 16));
  }
}

template <bool kFp8>
__device__ __forceinline__ void pf_put(uint8_t* tile, int kk, int sub, uint4 x) {
  uint8_t* row = tile + kk * 256;
  const int sw = pf_swz(kk);
  if constexpr (kFp8) {
    *reinterpret_cast<bf16x8_t*>(row + (((2 * sub) ^ sw) << 4)) = fp8x8w_to_bf16(x.x, x.y);
    *reinterpret_cast<bf16x8_t*>(row + (((2 * sub + 1) ^ sw) << 4)) = fp8x8w_to_bf16(x.z, x.w);
  } else {
    *reinterpret_cast<uint4*>(row + ((sub ^ sw) << 4)) = x;
  }
}

// The pieces of step i into a tile; rows of keys without a cache block (bad:
// the sequence has such entries) as zeros.
template <bool kFp8>
__device__ __forceinline__ void pf_store(const AttnArgs& a, int b, int i, int T, int wid,
                                         const PfTable& tab, bool bad,
                                         uint4 (&x)[PfStage<kFp8>::kPieces], uint8_t* tile) {
  using S = PfStage<kFp8>;
  const int lane = threadIdx.x & 63;
  const int row = wid * S::kRowsPerWave + lane / S::kLanesPerRow, sub = lane % S::kLanesPerRow;
  if (bad) {
    asm volatile("; missing blocks");
#pragma unroll
    for (int j = 0; j < S::kPieces; ++j) {
      const int key = min(i, T - 1) * kPfStep + ((j * S::kRowsPerPiece + row) & 32);
      if (pf_entry(a, b, key >> tab.shift, tab.nbt) < 0) x[j] = make_uint4(0, 0, 0, 0);
    }
  }
#pragma unroll
  for (int j = 0; j < S::kPieces; ++j) pf_put<kFp8>(tile, j * S::kRowsPerPiece + row, sub, x[j]);
}

// Infinities and NaN of a thread's pieces of V to zero; whether there were any.
template <bool kFp8>
__device__ __forceinline__ bool pf_finite(uint4 (&x)[PfStage<kFp8>::kPieces]) {
  // an all-ones exponent (bf16), or 0x7f / 0xff (e4m3fn), carries into the top bit
  constexpr uint32_t kAnd = kFp8 ? 0x7f7f7f7fu : 0x7f807f80u;
  constexpr uint32_t kAdd = kFp8 ? 0x01010101u : 0x00800080u;
  constexpr uint32_t kTop = kFp8 ? 0x80808080u : 0x80008000u;
  constexpr uint32_t kAll = kFp8 ? 0xffu : 0xffffu;
  uint32_t any = 0;
#pragma unroll
  for (int j = 0; j < PfStage<kFp8>::kPieces; ++j)
    any |= ((x[j].x & kAnd) + kAdd) | ((x[j].y & kAnd) + kAdd) | ((x[j].z & kAnd) + kAdd) |
           ((x[j].w & kAnd) + kAdd);
  if (!(any & kTop)) return false;
  auto zero = [&](uint32_t& w) {
    w &= ~(((((w & kAnd) + kAdd) & kTop) >> (kFp8 ? 7 : 15)) * kAll);
  };
#pragma unroll
  for (int j = 0; j < PfStage<kFp8>::kPieces; ++j) {
    zero(x[j].x);
    zero(x[j].y);
    zero(x[j].z);
    zero(x[j].w);
  }
  return true;
}

// Key splits of a call (kSplit): a list of pieces from the real lengths, as in
// the listed launch. A few new tokens behind a long cached prefix, in a call with
// a long prompt, or a prompt of few tiles behind one are otherwise one workgroup's
// chain of 1.4 (bf16) to 2.3 us (fp8) per 64 keys while the other CUs are done
// (200 tokens beside three sequences of one behind 8000, 32 heads over 8: 188 us,
// 16-row tiles 45, with splits 42; 300 tokens behind 8000: 193, 286, 85).
// A tile well longer than `len` steps is cut into equal pieces of about that
// many, len being the call's steps over `target` workgroups for a kv head and at
// least kPfMinSteps. target: one for a CU with bf16, whose streams fill the memory
// pipes (32 prompts of 32 tokens behind 2048: 73 us, two for a CU 94), two with
// FP8, half the bytes in flight (16 of 16 behind 8000: one for a CU 145 us,
// two 90).
// Partials go to the workspace, and the last workgroup of a tile to take its
// ticket merges them. A sequence that is cut has at most twice the pieces that its
// steps fill, so kPfPieces(target) slots and tickets for a kv head are enough.
// A kv head's workgroups take the pieces level by level, a sequence's i-th ones
// with the others' i-th, those of the sequence with the most keys early, and the
// workgroups without a piece come last: in between they held whole parts of the
// chip back (3000 tokens behind 4000 and three sequences of one behind 8000, fp8:
// 1115 us, 459 so).
constexpr int kPfMinSteps = 16;
constexpr int kPfPartO = kPfTileRows * kD;  // floats of one partial's outputs
constexpr size_t kPfSlotBytes = (kPfPartO + 2 * kPfTileRows) * sizeof(float);
__host__ __device__ constexpr int kPfPieces(int target) { return 2 * target; }

struct PfItem {
  int b, qt, piece, len, slot;  // sequence (-1: no piece), tile, its piece, most steps, slot of piece 0
  int q0, q1, k0, k1;
};

// The piece of workgroup idx of a kv head, by one wave (all waves of a workgroup
// the same): lane i holds sequence i.
__device__ __forceinline__ PfItem pf_item(const AttnArgs& a, int G, int qtiles, int target,
                                          int idx, int lane) {
  const int i = lane < a.B ? lane : a.B - 1;
  const int k0 = a.cu_k[i], k1 = a.cu_k[i + 1], q0 = a.cu_q[i], q1 = a.cu_q[i + 1];
  // (tiles past the declared maximum are not attended: the grid counts no workgroups
  // for them, and without the clamp they took those of other tiles' pieces, whose rows
  // stayed unwritten and whose tickets nonzero)
  const int rows = lane < a.B && q1 > q0 ? (q1 - q0) * G : 0;
  const int n = min((rows + kPfTileRows - 1) / kPfTileRows, qtiles);
  const int T = k1 > k0 ? (k1 - k0 + kPfStep - 1) / kPfStep : 0;
  constexpr int kMost = 1 << 24;  // per sequence, so that 64 of them add up (else: no splits)
  const int work = (int64_t)n * T < kMost ? n * T : kMost;
  const int total = __builtin_amdgcn_readlane(wave_scan<false>(work), 63);
  const int even = (total + target - 1) / target;
  const int len = __builtin_amdgcn_ballot_w64(work == kMost) ? kMost
                  : even > kPfMinSteps                       ? even
                                                             : kPfMinSteps;
  // (a tile little longer than len stays whole)
  const int c = max(list_ceil(T - len / 5, len, __builtin_amdgcn_rcpf((float)len)), 1);
  const int e = n * c, se = c > 1 ? e : 0;
  const int sincl = wave_scan<false>(se);
  PfItem it;
  it.b = -1;
  if (idx >= __builtin_amdgcn_readlane(wave_scan<false>(e), 63)) return it;
  // the idx-th piece, level by level; pieces in the levels before `lev`:
  const int most = __builtin_amdgcn_readlane(wave_scan<true>(e), 63);
  const int keys = __builtin_amdgcn_readlane(wave_scan<true>(T), 63);
  const int kl = __builtin_ctzll(__builtin_amdgcn_ballot_w64(T == keys));
  const bool down = 2 * __builtin_amdgcn_readlane(e, kl) >= most;
  auto before = [&](int lev) {
    const int x = down ? max(e - (most - lev), 0) : min(e, lev);
    return __builtin_amdgcn_readlane(wave_scan<false>(x), 63);
  };
  int lev = 0;
  for (int end = most; end - lev > 1;) {
    const int mid = (lev + end) >> 1;
    if (before(mid) <= idx)
      lev = mid;
    else
      end = mid;
  }
  const int at = down ? most - 1 - lev : lev;
  const uint64_t has = __builtin_amdgcn_ballot_w64(e > at);
  const int nth = __builtin_amdgcn_mbcnt_hi((uint32_t)(has >> 32),
                                            __builtin_amdgcn_mbcnt_lo((uint32_t)has, 0));
  const int pick = idx - before(lev);  // (in every lane: it sums over the wave)
  const int l = __builtin_ctzll(__builtin_amdgcn_ballot_w64(e > at && nth == pick));
  it.b = l;
  const int ln = __builtin_amdgcn_readlane(n, l);
  it.piece = at / ln;
  it.qt = at - it.piece * ln;
  it.len = len;
  it.slot = __builtin_amdgcn_readlane(sincl - se, l) + it.qt * __builtin_amdgcn_readlane(c, l);
  it.q0 = __builtin_amdgcn_readlane(q0, l);
  it.q1 = __builtin_amdgcn_readlane(q1, l);
  it.k0 = __builtin_amdgcn_readlane(k0, l);
  it.k1 = __builtin_amdgcn_readlane(k1, l);
  return it;
}

// The grid is (kv head fastest, then sequences, then query tiles from the last
// down): with 8 kv heads consecutive workgroups go to the 8 XCDs in turn, so a
// head's K and V stay in one XCD's L2, and the tiles with the most keys start
// first. kSplit: (kv head fastest, then the list of pieces).
template <bool kFp8, int kG, bool kSplit>
__global__ __launch_bounds__(kPfWaves * 64, 2) void k_prefill_attn(AttnArgs a, int qtiles,
                                                                   int target) {
  const int G = kG ? kG : a.G;
  __shared__ __attribute__((aligned(16))) uint8_t s_k[2 * kPfTileB];
  __shared__ __attribute__((aligned(16))) uint8_t s_v[2 * kPfTileB];
  __shared__ int s_nf;  // V of a masked step holds an infinity or NaN
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 31, h = lane >> 5;
  const int kvh = blockIdx.x % a.Hkv;
  const int rest = blockIdx.x / a.Hkv;
  int b, qt, first;
  TileRef t;
  PfItem it;
  if constexpr (kSplit) {
    it = pf_item(a, G, qtiles, target, rest, lane);
    if (it.b < 0) return;
    b = it.b;
    qt = it.qt;
    first = a.contig ? 0 : a.bt[(int64_t)b * a.bt_stride + min(lane, a.bt_width - 1)];
    t = tile_ref_of(b, kvh, qt, G, it.q0, it.q1, it.k0, it.k1);
  } else {
    b = rest % a.B;
    qt = qtiles - 1 - rest / a.B;
    // the first block-table entries go out with the sequence bounds
    first = a.contig ? 0 : a.bt[(int64_t)b * a.bt_stride + min(lane, a.bt_width - 1)];
    t = tile_ref(a, b, kvh, qt, G);
  }
  const int r0 = qt * kPfTileRows;
  if (r0 >= t.rows) return;

  // keys visible to the workgroup's last row, and to the wave's rows
  const int rl = min(r0 + kPfTileRows, t.rows) - 1;
  int khi = min(t.Lk, t.Lk - t.Lq + rl / G + 1);
  khi = khi > 0 ? khi : 0;
  const int wr0 = r0 + wid * 32;
  const int kfull = min(khi, t.Lk - t.Lq + wr0 / G + 1);  // below it: visible to all its rows
  const int kfull_all = min(khi, t.Lk - t.Lq + r0 / G + 1);  // visible to all the tile's rows
  const bool act = wr0 < t.rows;  // a wave without rows only moves its share of K and V

  // this workgroup's steps [i0, T) of the tile's, in pieces of `steps`
  int T = (khi + kPfStep - 1) / kPfStep, i0 = 0, pieces = 1;
  if constexpr (kSplit) {
    pieces = max((T - it.len / 5 + it.len - 1) / it.len, 1);
    if (pieces > 1) {
      const int steps = (T + pieces - 1) / pieces;
      pieces = (T + steps - 1) / steps;
      i0 = it.piece * steps;
      T = min(T, i0 + steps);
    }
    if (it.piece >= pieces) return;
  }

  // this lane's query row
  const int r = wr0 + n;
  const bool r_ok = r < t.rows;
  const int qi = r_ok ? r / G : 0;
  const int qh = kvh * G + (r_ok ? r % G : 0);
  const int lim_r = r_ok ? t.Lk - t.Lq + qi : -1;  // its last visible key
  bf16x8_t qv[8];
  {
    const uint16_t* qp = a.q + (int64_t)(t.qs + qi) * a.q_st + (int64_t)qh * a.q_sh + h * 8;
#pragma unroll
    for (int dc = 0; dc < 8; ++dc)
      qv[dc] = u4_to_bf16x8(*reinterpret_cast<const uint4*>(qp + dc * 16));
  }

  // a visible key whose block-table entry is no cache block is skipped (bad)
  PfTable tab;
  tab.shift = a.contig ? 30 : a.bs_shift;
  tab.s_blk = a.contig ? 0 : a.c_sb;
  tab.nbt = khi > 0 ? ((khi - 1) >> tab.shift) + 1 : 0;
  tab.base = 0;
  tab.entry = (a.contig || (lane < min(tab.nbt, a.bt_width) && first < a.num_blocks)) ? first : -1;
  bool bad = __builtin_amdgcn_ballot_w64(lane < tab.nbt && tab.entry < 0) != 0;
  for (int i = 64; i < tab.nbt; i += 64)
    bad |= __builtin_amdgcn_ballot_w64(i + lane < tab.nbt && pf_entry(a, b, i + lane, tab.nbt) < 0) != 0;
  if constexpr (kSplit) {
    const int e0 = (i0 * kPfStep) >> tab.shift;
    if (e0 >= 64) {
      tab.base = e0 & ~63;
      tab.entry = pf_entry(a, b, tab.base + lane, tab.nbt);
    }
  }
  const int64_t head = (int64_t)kvh * a.c_sh + (a.contig ? (int64_t)t.ks * a.c_st : 0);
  const uint8_t* kcache = a.kc + head * (kFp8 ? 1 : 2);
  const uint8_t* vcache = a.vc + head * (kFp8 ? 1 : 2);
  const uint32_t rowb = (uint32_t)(a.c_st * (kFp8 ? 1 : 2));

  // operand addresses within a tile: K row n (+ 32), V rows 4h + n16 / 4 (+ 8,
  // + 16, ...) at the d-block's chunks
  int ka_off[8], va_off[2][4];
#pragma unroll
  for (int dc = 0; dc < 8; ++dc) ka_off[dc] = n * 256 + (((2 * dc + h) ^ pf_swz(n)) << 4);
#pragma unroll
  for (int h2 = 0; h2 < 2; ++h2)
#pragma unroll
    for (int db = 0; db < 4; ++db) {
      const int key = 8 * h2 + 4 * h + ((lane & 15) >> 2);
      const int c = 4 * db + 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
      va_off[h2][db] = key * 256 + ((c ^ pf_swz(key)) << 4) + ((lane & 1) << 3);
    }

  float m = -INFINITY, lsum = 0.0f;
  f32x16_t oacc[4];
#pragma unroll
  for (int db = 0; db < 4; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) oacc[db][i] = 0.0f;

  f32x16_t sc[2];
  bf16x8_t pb[2][2], pl[2];
  // S^T of step ws: sc[kb][i] is row n, key ws + 32 kb + 8 (i / 4) + 4h + i % 4
  auto scores = [&](const uint8_t* tk) __attribute__((always_inline)) {
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int i = 0; i < 16; ++i) sc[kb][i] = 0.0f;
#pragma unroll
    for (int dc = 0; dc < 8; ++dc)
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        const bf16x8_t kf = u4_to_bf16x8(
            *reinterpret_cast<const uint4*>(tk + kb * (32 * 256) + ka_off[dc]));
        sc[kb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qv[dc], sc[kb], 0, 0, 0);
      }
  };
  // fine (masked steps): with what bf16 leaves of the first 32 keys' probabilities
  // (pl). Rows with few keys have them all there, and with 32 rows to a wave fewer
  // of a row's probabilities are exact powers of two than when eight waves share its
  // keys. The error against float64 is so no larger than in 16-row tiles: unpaged
  // prompts of 61 to 1021 tokens 1.83e-3, 1.95e-3 in those, 2.04e-3 without (which
  // took 46.5 us for them, 48.2 so; 6301 tokens alike).
  auto values = [&](const uint8_t* tv, auto fine) __attribute__((always_inline)) {
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int db = 0; db < 4; ++db) {
          union {
            v4i16_t x[2];
            bf16x8_t v;
          } vf;
#pragma unroll
          for (int h2 = 0; h2 < 2; ++h2)
            vf.x[h2] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (HS_LDS v4i16_t*)(tv + (kb * 32 + c * 16) * 256 + va_off[h2][db]));
          oacc[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf.v, pb[kb][c], oacc[db], 0, 0, 0);
          if (decltype(fine)::value && kb == 0)
            oacc[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf.v, pl[c], oacc[db], 0, 0, 0);
        }
  };
  auto softmax = [&](int ws, auto fine) __attribute__((always_inline)) {
    if (ws + kPfStep > kfull || bad) {
      asm volatile("; masked step");
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        const bool gone = bad && pf_entry(a, b, (ws + 32 * kb) >> tab.shift, tab.nbt) < 0;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int key = ws + 32 * kb + 8 * (i >> 2) + 4 * h + (i & 3);
          if (gone || key >= khi || key > lim_r) sc[kb][i] = -INFINITY;
        }
      }
    }
    float mloc = -INFINITY;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int i = 0; i < 16; ++i) mloc = fmaxf(mloc, sc[kb][i]);
    {
      const auto x = __builtin_amdgcn_permlane32_swap(__float_as_uint(mloc),
                                                      __float_as_uint(mloc), false, false);
      mloc = fmaxf(__uint_as_float(x[0]), __uint_as_float(x[1])) * a.scale_log2;
    }
    const bool up = mloc > m + kRefSlack;
    if (__builtin_amdgcn_ballot_w64(up)) {
      const float m_new = up ? mloc : m;
      if (__builtin_amdgcn_ballot_w64(up && m != -INFINITY)) {
        const float alpha = (m_new == m) ? 1.0f : __builtin_amdgcn_exp2f(m - m_new);
        lsum *= alpha;
#pragma unroll
        for (int db = 0; db < 4; ++db) oacc[db] *= alpha;
      }
      m = m_new;
    }
    const float base = (m == -INFINITY) ? 0.0f : m;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        union {
          uint16_t u[8];
          bf16x8_t v;
        } pk, lo;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float p =
              __builtin_amdgcn_exp2f(__builtin_fmaf(sc[kb][8 * c + e], a.scale_log2, -base));
          lsum += p;
          pk.u[e] = f32_to_bf16_rne(p);
          if (decltype(fine)::value && kb == 0)
            lo.u[e] = f32_to_bf16_rne(p - __uint_as_float((uint32_t)pk.u[e] << 16));
        }
        pb[kb][c] = pk.v;
        if (decltype(fine)::value && kb == 0) pl[c] = lo.v;
      }
    // made here, not sunk into the matrix work below (that spills)
    asm volatile("" : "+v"(lsum), "+v"(pb[0][0]), "+v"(pb[0][1]), "+v"(pb[1][0]), "+v"(pb[1][1]));
    if (decltype(fine)::value) asm volatile("" : "+v"(pl[0]), "+v"(pl[1]));
  };

  // Step i: scores(i), softmax(i), values(i). K(i) and V(i) sit in buffers
  // (i - i0) % 2. Iteration i multiplies V(i) and K(i + 1), loads V(i + 1) and K(i +
  // 2) at its start and stores them at its end into the buffers of V(i - 1)
  // and K(i), whose last reads ended at the barrier before; the barrier after
  // the stores makes them readable.
  using S = PfStage<kFp8>;
  uint4 kx[S::kPieces], vx[S::kPieces];
  auto load = [&](const uint8_t* cache, const PfStep& p, uint4 (&x)[S::kPieces]) __attribute__((always_inline)) {
    pf_load<kFp8>(cache, p, rowb, wid, x);
  };
  auto store = [&](int i, uint4 (&x)[S::kPieces], uint8_t* tile) __attribute__((always_inline)) {
    pf_store<kFp8>(a, b, i, T, wid, tab, bad, x, tile);
  };
  // P = 0 does not keep an infinity or NaN of V out of a row that does not see its
  // key, so those of the masked steps stay out of the products and are added to the
  // rows that do see them after the last one. The iterations that store a masked
  // step's V are a loop of their own: the branch in the one loop cost 7% (prompts of
  // up to 1021 tokens).
  const int masked = max(kfull_all, 0) / kPfStep;  // the first masked step
  if (i0 < T) {
    if (tid == 0) s_nf = 0;
    PfStep vstep = pf_step(a, b, i0, T, khi, tab);  // the step of the next V rows
    load(kcache, vstep, kx);
    load(vcache, vstep, vx);
    store(i0, kx, s_k);
    vstep = pf_step(a, b, i0 + 1, T, khi, tab);
    load(kcache, vstep, kx);
    lds_barrier();
    if (act) scores(s_k);
    store(i0 + 1, kx, s_k + kPfTileB);
    if (i0 >= masked && pf_finite<kFp8>(vx)) s_nf = 1;
    store(i0, vx, s_v);
    lds_barrier();
    int cur = 0;
    auto iterate = [&](int i, auto check) __attribute__((always_inline)) {
      const int oth = kPfTileB - cur;
      load(vcache, vstep, vx);
      vstep = pf_step(a, b, i + 2, T, khi, tab);
      load(kcache, vstep, kx);
      if (act) {
        softmax(i * kPfStep, check);
        values(s_v + cur, check);
        scores(s_k + oth);
        // LDS reads run ahead of the matrix instructions by kPfAhead operands
        __builtin_amdgcn_sched_group_barrier(0x100, kPfAhead, 0);
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        }
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
      }
      store(i + 2, kx, s_k + cur);
      if (decltype(check)::value && pf_finite<kFp8>(vx)) s_nf = 1;
      store(i + 1, vx, s_v + oth);
      lds_barrier();
      cur ^= kPfTileB;
    };
    int i = i0;
    for (; i < min(masked - 1, T - 1); ++i) iterate(i, std::false_type{});
    for (; i < T - 1; ++i) iterate(i, std::true_type{});
    if (act) {
      softmax((T - 1) * kPfStep, std::true_type{});
      values(s_v + cur, std::true_type{});
    }
    if (__builtin_amdgcn_readfirstlane(s_nf)) {
      const int from = max(i0 * kPfStep, kfull_all / kPfStep * kPfStep);
      const int end = min(min(khi, T * kPfStep), lim_r + 1);
#pragma unroll 1
      for (int key = from; key < end; ++key) {
        const int e = key >> tab.shift, blk = pf_entry(a, b, e, tab.nbt);
        if (blk < 0) continue;
        const uint8_t* row = vcache + ((int64_t)blk * tab.s_blk +
                                       (int64_t)(key - (e << tab.shift)) * a.c_st) * (kFp8 ? 1 : 2);
#pragma unroll
        for (int db = 0; db < 4; ++db)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const int d = db * 32 + 8 * (i >> 2) + 4 * h + (i & 3);
            const uint32_t w = kFp8 ? row[d] : reinterpret_cast<const uint16_t*>(row)[d];
            if (kFp8 ? (w & 0x7f) == 0x7f : (w & 0x7f80) == 0x7f80)
              oacc[db][i] += kFp8 ? NAN : __uint_as_float(w << 16);
          }
      }
    }
  }

  {
    const auto x = __builtin_amdgcn_permlane32_swap(__float_as_uint(lsum), __float_as_uint(lsum),
                                                    false, false);
    lsum = __uint_as_float(x[0]) + __uint_as_float(x[1]);
  }
  if constexpr (kSplit) {
    if (pieces > 1) {
      // A partial is laid out as its lanes hold it, 16 bytes a lane side by side,
      // so the workgroup that merges reads its own places back; agent-scope
      // stores and loads, as in merge_tile.
      __shared__ int s_last;
      const int piece = it.piece;
      const int64_t slot0 = (int64_t)kvh * kPfPieces(target) + it.slot;
      const int at = wid * 64 + lane, row = wid * 32 + n;
      if (r_ok) {
        float* po = a.part_o + (slot0 + piece) * kPfPartO + at * 4;
#pragma unroll
        for (int db = 0; db < 4; ++db)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            part_store4<true>(po + (db * 4 + j) * (kPfWaves * 256), oacc[db][4 * j],
                              oacc[db][4 * j + 1], oacc[db][4 * j + 2], oacc[db][4 * j + 3]);
        if (h == 0)
          part_store2<true>(a.part_ml + ((slot0 + piece) * kPfTileRows + row) * 2, m, lsum);
      }
      unsigned* ticket = a.tickets + slot0;
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (tid == 0) {
        const unsigned prev =
            __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        s_last = prev + 1 == (unsigned)pieces;
      }
      __syncthreads();
      if (!s_last) return;
      if (tid == 0) __hip_atomic_store(ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (!r_ok) return;
      m = -INFINITY;
      for (int s = 0; s < pieces; ++s)
        m = fmaxf(m, part_load2<true>(a.part_ml + ((slot0 + s) * kPfTileRows + row) * 2).x);
      const float base = (m == -INFINITY) ? 0.0f : m;
      lsum = 0.0f;
#pragma unroll
      for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) oacc[db][i] = 0.0f;
      for (int s = 0; s < pieces; ++s) {  // in order: the same bits whoever merges
        const float2 ml = part_load2<true>(a.part_ml + ((slot0 + s) * kPfTileRows + row) * 2);
        const float f = __builtin_amdgcn_exp2f(ml.x - base);
        lsum += ml.y * f;
        const float* po = a.part_o + (slot0 + s) * kPfPartO + at * 4;
#pragma unroll
        for (int db = 0; db < 4; ++db)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const float* p = po + (db * 4 + j) * (kPfWaves * 256);
            const float2 x = part_load2<true>(p), y = part_load2<true>(p + 2);
            oacc[db][4 * j] += x.x * f;
            oacc[db][4 * j + 1] += x.y * f;
            oacc[db][4 * j + 2] += y.x * f;
            oacc[db][4 * j + 3] += y.y * f;
          }
      }
    }
  }
  if (!r_ok) return;
  const float inv = (lsum > 0.0f) ? a.v_scale / lsum : 0.0f;
  uint16_t* op = a.out + (int64_t)(t.qs + qi) * a.o_st + (int64_t)qh * a.o_sh + 4 * h;
#pragma unroll
  for (int db = 0; db < 4; ++db)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t w0 = (uint32_t)f32_to_bf16_rne(oacc[db][4 * j] * inv) |
                          ((uint32_t)f32_to_bf16_rne(oacc[db][4 * j + 1] * inv) << 16);
      const uint32_t w1 = (uint32_t)f32_to_bf16_rne(oacc[db][4 * j + 2] * inv) |
                          ((uint32_t)f32_to_bf16_rne(oacc[db][4 * j + 3] * inv) << 16);
      *reinterpret_cast<uint2*>(op + db * 32 + 8 * j) = make_uint2(w0, w1);
    }
}

// How the prompt kernel serves a call.
struct PfPlan {
  bool use;
  int qtiles, target;  // target 0: no key splits
};
constexpr int64_t kPfMaxGrid = (1 << 24) - 1;  // workgroups of 256 threads a launch takes
// The rule (tokens: the call's query tokens, -1 where the caller does not say; a
// batch's prompts are then taken to be half the longest one on average):
// - a sequence has 32 rows on average. One of 28 rows costs here what it costs in
//   two 16-row tiles; batches of mostly shorter ones are left to that launch,
//   which streams their keys faster (fp8, 100 tokens and 31 sequences of 4, all
//   behind 4000 keys: 85 us, 115 here). Where the balanced launch does not take
//   the call (more than kSkMaxTiles tiles), the 16-row grid that does is the
//   slower one at any length (400 tokens, 63 sequences of one: 318 us, 64 here).
// - with key splits, 360 16-row tiles: below, the balanced launch has as few
//   rounds to go and no merge of 128-row partials (32 heads over 8, bf16, 4 x 32
//   tokens behind 2048 keys, 280 tiles: 31 us, 36 here; 8 x 16 behind 2048, 304:
//   31, 37 here; 10 x 16 behind 2048, 380: 67, 39 here, behind 8000 207 and 82).
// - without, 640: a tile is then one chain of 1.4 us per 64 keys, a 16-row tile
//   2.2 (fp8) to 2.8 ns of the whole GPU's time. And only where no sequence can be
//   a long chain by itself: one sequence, keys no longer than the longest prompt
//   or few, or more sequences than a wave holds (whose tiles fill the CUs).
constexpr int kPfRows = 32, kPfTiles = 360, kPfTilesWhole = 640;

// Workspace that lets a call of the prompt kernel split its keys.
static size_t prefill_workspace(int Hkv, int cus) {
  const int target = (2 * cus + Hkv - 1) / Hkv;
  return kTicketBytes + (size_t)Hkv * kPfPieces(target) * kPfSlotBytes;
}

// scratch: the call's launch in 16-row tiles would hold partials in the workspace,
// and there is one. balanced: that launch is the balanced one.
static PfPlan prefill_plan(const AttnArgs& a, int tokens, int max_seqlen_q, int max_seqlen_k,
                           bool scratch, size_t workspace_bytes, bool balanced, int cus) {
  const int64_t full = (int64_t)max_seqlen_q * a.G;
  const int64_t qtiles = (full + kPfTileRows - 1) / kPfTileRows;
  const int64_t pairs = (int64_t)a.B * a.Hkv;
  const int target = ((a.fp8 ? 2 : 1) * cus + a.Hkv - 1) / a.Hkv;
  PfPlan p{false, (int)qtiles, 0};
  const int64_t rows = tokens >= 0 ? (int64_t)tokens * a.G : a.B > 1 ? a.B * full / 2 : full;
  if ((!a.contig && a.bs_shift < 5) || (qtiles * a.B + target) * a.Hkv > kPfMaxGrid) return p;
  if (full < kPfRows || (balanced && rows < (int64_t)kPfRows * a.B)) return p;
  // 16-row tiles: a sequence's last one is part empty
  const int64_t tiles = (rows / kRows + 3 * (int64_t)a.B / 4) * a.Hkv;
  // as many pieces as the workspace holds, one for two CUs at least; calls whose
  // keys are one piece anyway take none
  int64_t fit = 0;
  if (scratch && a.B <= 64 && workspace_bytes > kTicketBytes &&
      max_seqlen_k > kPfMinSteps * kPfStep && (a.B > 1 || qtiles < target)) {
    const size_t one = (size_t)a.Hkv * kPfPieces(1) * kPfSlotBytes;
    fit = std::min<int64_t>(kTicketSlots / (a.Hkv * kPfPieces(1)),
                            (int64_t)((workspace_bytes - kTicketBytes) / one));
    fit = std::min<int64_t>(fit, target);
  }
  if (4 * fit >= target) {
    p.use = tiles >= kPfTiles;
    p.target = (int)fit;
  } else {
    p.use = a.qtiles * pairs >= kPfTilesWhole &&
            (a.B == 1 || a.B > 64 || max_seqlen_k <= max_seqlen_q ||
             max_seqlen_k <= kPfMinSteps * kPfStep);
  }
  return p;
}

template <bool kFp8, bool kSplit>
static void launch_prefill(const AttnArgs& a, const PfPlan& p, hipStream_t s) {
  const int64_t entries = (int64_t)p.qtiles * a.B + (kSplit ? p.target : 0);
  const dim3 grid((unsigned)(entries * a.Hkv)), block(kPfWaves * 64);
  switch (a.G) {
    case 2: hipLaunchKernelGGL((k_prefill_attn<kFp8, 2, kSplit>), grid, block, 0, s, a, p.qtiles, p.target); break;
    case 4: hipLaunchKernelGGL((k_prefill_attn<kFp8, 4, kSplit>), grid, block, 0, s, a, p.qtiles, p.target); break;
    default: hipLaunchKernelGGL((k_prefill_attn<kFp8, 0, kSplit>), grid, block, 0, s, a, p.qtiles, p.target); break;
  }
}

}  // namespace hs

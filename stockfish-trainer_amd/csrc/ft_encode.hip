// Feature-index encoder: chess positions -> the FT's sparse index rows
// (HalfKAv2_hm, Full_Threats and their composition), on the GPU.
//
// Replaces the reference's per-position index extraction
// (src/rust/feature_extraction.rs: FeatureSet::fill_feature_indices_sparse
// :209-236, fill_row_from_position_without_values :442-477, the HalfKAv2_hm
// indices :389-402, 677-685 and the Full_Threats indices :572-675, 687-833),
// which the reference runs on CPU threads and ships to the GPU as int32 slabs.
// Here the positions travel (65 bytes each) and the slabs are produced in HBM.
//
// Conventions (those of the sfbinpack crate the reference is written
// against): square a1 = 0 .. h8 = 63; piece id = 2 * type + color, types pawn,
// knight, bishop, rook, queen, king = 0..5, white = 0; bitboards are walked
// from the lowest square up.  board[64] holds a piece id or 255 (empty).
//
// One wave per position, a few consecutive positions per wave.  First a lane per
// square: twelve ballots give the bitboards (uniform, so scalar), a lane's rank
// among them its piece's place in the threat order, and HalfKAv2_hm's features
// are one lane each.  Then a lane per (perspective, piece): the pieces of a
// perspective stand in the order the reference walks them (own colour first,
// then by type and square), so a feature's slot is a prefix sum over lanes of
// the pieces' target counts (four ballots, a count is at most 8) -- only pawns,
// walked by direction before square, need a count per direction.  Rows are
// filled in LDS and stored with 16-byte stores.  Bound by instruction issue
// (about 700 vector instructions a position; the rows' 1.3 KB take 17 us per
// 65 536 positions): Full_Threats+HalfKAv2_hm 180 -> 75 us against a thread per
// (position, perspective), whose waves walked 64 unlike positions in lockstep.
#include "common.h"

namespace sft {

namespace {

constexpr int kPawn = 0, kKnight = 1, kBishop = 2, kRook = 3, kQueen = 4, kKing = 5;
constexpr int kHalfkaInputs = 24576, kHalfkaMax = 32, kThreatInputs = 60720, kThreatMax = 128;

// src/rust/feature_extraction.rs:27-28: valid attacked (colour, type) pairs of an attacker type.
constexpr int kNumValidTargets[6] = {6, 10, 8, 8, 10, 0};

// King bucket of an oriented king square (files e-h after orientation):
// (7 - rank) * 4 + (7 - file) (src/rust/feature_extraction.rs:21-25).
__device__ __forceinline__ int king_bucket(int sq) { return (7 - (sq >> 3)) * 4 + (7 - (sq & 7)); }

// ---- tables (built by the compiler, copied to LDS by each workgroup) ----
// Attackers by kind: pawns of each colour, then knight .. queen.
constexpr int kKinds = 6;
__host__ __device__ constexpr int kind_of(int type, int color) { return type == kPawn ? color : type + 1; }
constexpr uint64_t square_bit(int f, int r) {
  return f >= 0 && f < 8 && r >= 0 && r < 8 ? (uint64_t)1 << (r * 8 + f) : 0;
}
// Squares from `from` in direction (df, dr), to the edge.
constexpr uint64_t ray(int from, int df, int dr) {
  uint64_t a = 0;
  for (int i = 1; i < 8; ++i) a |= square_bit((from & 7) + i * df, (from >> 3) + i * dr);
  return a;
}
constexpr int bit_count(uint64_t x) {
  int n = 0;
  for (; x; x &= x - 1) ++n;
  return n;
}
struct alignas(16) EncodeTables {
  uint64_t line[4][64];       // rank, file, diagonals through a square, without it
  uint64_t mask[kKinds][64];  // attack set on an empty board (pawns: captures and push, :723-733)
  uint16_t off[kKinds][64];   // features of a kind and target before those of a from-square (threat_feature_calc, :795-833)
  int size[kKinds];           // ... of all from-squares
  int base[2][5];             // first feature of a (colour, type) attacker: colour outer, type inner (:800-828)
  constexpr EncodeTables() : line{}, mask{}, off{}, size{}, base{} {
    for (int s = 0; s < 64; ++s) {
      const int f = s & 7, r = s >> 3;
      line[0][s] = ray(s, 1, 0) | ray(s, -1, 0);
      line[1][s] = ray(s, 0, 1) | ray(s, 0, -1);
      line[2][s] = ray(s, 1, 1) | ray(s, -1, -1);
      line[3][s] = ray(s, 1, -1) | ray(s, -1, 1);
      for (int c = 0; c < 2; ++c) {
        const int u = c == 0 ? r + 1 : r - 1;
        mask[c][s] = r == 0 || r == 7 ? 0 : square_bit(f - 1, u) | square_bit(f, u) | square_bit(f + 1, u);
      }
      for (int d = 1; d <= 2; ++d)
        mask[kind_of(kKnight, 0)][s] |= square_bit(f + d, r + 3 - d) | square_bit(f - d, r + 3 - d) |
                                        square_bit(f + d, r - 3 + d) | square_bit(f - d, r - 3 + d);
      mask[kind_of(kBishop, 0)][s] = line[2][s] | line[3][s];
      mask[kind_of(kRook, 0)][s] = line[0][s] | line[1][s];
      mask[kind_of(kQueen, 0)][s] = mask[kind_of(kBishop, 0)][s] | mask[kind_of(kRook, 0)][s];
    }
    for (int k = 0; k < kKinds; ++k)
      for (int s = 0; s < 64; ++s) {
        off[k][s] = (uint16_t)size[k];
        size[k] += bit_count(mask[k][s]);
      }
    int n = 0;
    for (int c = 0; c < 2; ++c)
      for (int t = 0; t < 5; ++t) {
        base[c][t] = n;
        n += kNumValidTargets[t] * size[kind_of(t, c)];
      }
  }
};
constexpr EncodeTables kTables{};
static_assert(kTables.base[1][kQueen] + kNumValidTargets[kQueen] * kTables.size[kind_of(kQueen, 1)] == kThreatInputs,
              "the threat features of all attackers");
static_assert(sizeof(EncodeTables) % 16 == 0, "copied in 16-byte pieces");
__device__ const EncodeTables kDeviceTables{};

__device__ __forceinline__ uint64_t rev64(uint64_t x) { return __builtin_bitreverse64(x); }
__device__ __forceinline__ int lsb64(uint64_t x) { return __ffsll((unsigned long long)x) - 1; }
// Bits of x below bit n.
__device__ __forceinline__ int popc_under(uint64_t x, int n) {
  const uint32_t part = (1u << (n & 31)) - 1u;
  const uint32_t lo = (uint32_t)x, hi = (uint32_t)(x >> 32);
  return n < 32 ? __popc(lo & part) : __popc(lo) + __popc(hi & part);
}
// Lanes 0 .. n-1.
__device__ __forceinline__ uint64_t lanes_below(int n) { return n >= 64 ? ~0ull : (1ull << n) - 1; }

// Sliding attacks along one line: occupied squares minus twice the slider, from
// either end (o ^ (o - 2r)); occ and rocc are the occupancy and its reverse.
__device__ __forceinline__ uint64_t line_attacks(uint64_t m, uint64_t occ, uint64_t two, uint64_t rtwo) {
  const uint64_t o = occ & m;
  return ((o - two) ^ rev64(rev64(o) - rtwo)) & m;
}

struct Encoding {
  int ncomp;
  int comp[2];  // 1 = Full_Threats, 2 = HalfKAv2_hm, in feature-set order
  int K;
};

// The wave's position: uniform bitboards by piece id, and per-wave LDS.
struct WavePosition {
  uint64_t bb[12], occ;
  int ksq[2];        // king squares (-1: none)
  int count[2];      // pieces by colour
  const uint8_t *board;          // piece id per square
  const uint16_t *pieces[2];     // per perspective, in its walking order: square | id << 8
};

// Full_Threats features (fill_full_threat_feature_indices_sparse, :572-675;
// full_threat_index, :687-737) into rows[perspective], slots from base on, the
// first kThreatMax of each row; offset is added to every feature.  total[p]:
// all features of perspective p.  BOTH: lanes 0-31 hold perspective 0's pieces
// and 32-63 perspective 1's (up to 32 pieces); else all 64 lanes `only`'s.
template <bool BOTH>
__device__ __forceinline__ void threat_rows(const EncodeTables &T, const WavePosition &w, int only, int32_t *rows,
                                            int K, int base, int offset, int *total) {
  const int lane = lane_id();
  const int p = BOTH ? lane >> 5 : only;  // uniform unless BOTH
  const int i = BOTH ? lane & 31 : lane;
  const int np = w.count[0] + w.count[1];
  const bool live = i < np;
  const unsigned e = live ? (p == 0 ? w.pieces[0] : w.pieces[1])[i] : 0u;
  const int from = e & 0xff, pc = (int)(e >> 8), type = pc >> 1, color = pc & 1;
  const bool attacker = live && type != kKing;
  // o: the perspective's orientation, as the threat features' own
  auto orient = [&](int q) { return ((w.ksq[q] & 7) >= 4 ? 7 : 0) ^ (q == 1 ? 56 : 0); };
  const int o = BOTH ? (p == 0 ? orient(0) : orient(1)) : orient(only);
  const bool enemy_persp = (color != p);

  // targets on the board: valid attacked types, less those of the attacker's own
  // type that another square counts (:711-718)
  const uint64_t pawns = w.bb[0] | w.bb[1], knights = w.bb[2] | w.bb[3], rooks = w.bb[6] | w.bb[7];
  const uint64_t minor = pawns | knights | w.bb[4] | w.bb[5] | rooks, major = minor | w.bb[8] | w.bb[9];
  uint64_t targets = 0;
  {
    const uint64_t r = 1ull << from, two = r << 1, rtwo = rev64(r) << 1;
    const uint64_t orth = line_attacks(T.line[0][from], w.occ, two, rtwo) | line_attacks(T.line[1][from], w.occ, two, rtwo);
    const uint64_t diag = line_attacks(T.line[2][from], w.occ, two, rtwo) | line_attacks(T.line[3][from], w.occ, two, rtwo);
    uint64_t att = type == kKnight ? T.mask[kind_of(kKnight, 0)][from] : 0ull;
    att |= (type == kRook || type == kQueen) ? orth : 0ull;
    att |= (type == kBishop || type == kQueen) ? diag : 0ull;
    // squares of oriented index above the attacker's, back on the board: bits of
    // each byte reversed (o & 7), bytes reversed (o & 56)
    uint64_t above = ~0ull << (from ^ o);  // the square itself is no target
    const uint64_t swapped = __builtin_bswap64(above);
    above = (o & 56) ? swapped : above;
    const uint64_t flipped = __builtin_bswap64(rev64(above));
    above = (o & 7) ? flipped : above;
    const uint64_t own_type = type == kKnight ? knights : type == kBishop ? (w.bb[4] | w.bb[5])
                              : type == kRook ? rooks : (w.bb[8] | w.bb[9]);
    targets = att & (type == kKnight || type == kQueen ? major : minor) & ~(own_type & above);
    targets = attacker && type != kPawn ? targets : 0ull;
  }
  // pawns: captures towards h, towards a (as White sees them), pushes; an enemy
  // pawn is a target only of the pawns that walk towards the perspective's side
  uint64_t pv[3] = {0, 0, 0};  // ballots: lanes whose pawn has target k
  int pto[3];
  bool has[3];
  {
    const uint64_t own_pawns = color == 0 ? w.bb[0] : w.bb[1];
    const uint64_t pt = enemy_persp ? pawns : own_pawns;
    const uint64_t captured = pt | knights | rooks;
    const int f = from & 7, step = color == 0 ? 1 : -1;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      pto[k] = from + step * (k == 0 ? 9 : k == 1 ? 7 : 8);
      const int edge = k == 0 ? (color == 0 ? 7 : 0) : (color == 0 ? 0 : 7);
      has[k] = attacker && type == kPawn && (unsigned)pto[k] < 64u && (k == 2 || f != edge) &&
               (((k == 2 ? pt : captured) >> (pto[k] & 63)) & 1);
      pv[k] = ballot(has[k]);
    }
  }
  const int cnt = type == kPawn ? (int)has[0] + (int)has[1] + (int)has[2] : __popcll(targets);  // at most 8

  // prefix sums of cnt over the perspective's lanes, totals and the first colour's total
  int start = 0, sum[2] = {0, 0}, own[2] = {0, 0};
  const int first = BOTH ? 32 : 0;  // perspective 1's first lane
  const uint64_t own0 = lanes_below(w.count[0]), own1 = lanes_below(w.count[1]) << first;
#pragma unroll
  for (int j = 3; j >= 0; --j) {
    const uint64_t b = ballot((cnt >> j) & 1);
    start = 2 * start + popc_below(b);
    sum[0] = 2 * sum[0] + __popcll(BOTH ? b & 0xffffffffull : b);
    sum[1] = 2 * sum[1] + __popcll(BOTH ? b >> 32 : b);
    own[0] = 2 * own[0] + __popcll(b & own0);
    own[1] = 2 * own[1] + __popcll(b & own1);
  }
  if (BOTH && p == 1) start -= sum[0];
  if (BOTH) total[0] = sum[0], total[1] = sum[1];
  else total[only] = sum[only];

  int32_t *row = rows + p * K + base;
  const int limit = kThreatMax;
  // the feature of target `to` apart from the attacker's share
  const int ppc = color ^ p;  // the attacker's colour as the perspective sees it
  const int pkind = type == kKing ? 0 : kind_of(type, ppc);
  const int pfrom = from ^ o;
  const uint64_t mask = T.mask[pkind][pfrom];
  const int size = T.size[pkind];
  const int half = type == kPawn ? 3 : type == kKnight || type == kQueen ? 5 : 4;
  const int share = offset + T.base[ppc][type == kKing ? 0 : type] + (int)T.off[pkind][pfrom];
  auto put = [&](int slot, int to) {
    const int a = w.board[to];
    const int mapped = (type == kPawn && (a >> 1) == kRook) ? 2 : a >> 1;
    if (slot < limit) row[slot] = share + (((a & 1) ^ p) * half + mapped) * size + popc_under(mask, to ^ o);
  };
  // pawns of a colour by direction: after the colours before, the directions
  // before, and the lanes below
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    int lead[2][2];  // [perspective][second colour]: its first slot less the counted lanes below its own
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const uint64_t mine = q == 0 ? own0 : own1;
      const uint64_t under = q == 0 ? 0ull : lanes_below(first);  // lanes before the perspective's
#pragma unroll
      for (int second = 0; second < 2; ++second) {
        const uint64_t below = second ? under | mine : under;
        const uint64_t half_lanes = BOTH ? (q == 0 ? 0xffffffffull : ~0xffffffffull) : ~0ull;
        const uint64_t block = second ? half_lanes & ~mine : mine;
        int n = second ? own[q] : 0;
        if (k > 0) n += __popcll(pv[0] & block);
        if (k > 1) n += __popcll(pv[1] & block);
        lead[q][second] = n - __popcll(pv[k] & below);
      }
    }
    const int l0 = enemy_persp ? lead[0][1] : lead[0][0], l1 = enemy_persp ? lead[1][1] : lead[1][0];
    if (has[k]) put((p == 0 ? l0 : l1) + popc_below(pv[k]), pto[k]);
  }
  for (int slot = start; targets; targets &= targets - 1, ++slot) put(slot, lsb64(targets));
}

template <bool THREATS>
__global__ __launch_bounds__(kBlock) void encode_kernel(const uint8_t *__restrict__ boards,
                                                        const uint8_t *__restrict__ stm, int64_t B, Encoding enc,
                                                        int per_wave, int32_t *__restrict__ white,
                                                        int32_t *__restrict__ black, float *__restrict__ us,
                                                        int64_t *__restrict__ psqt, int64_t *__restrict__ ls,
                                                        int32_t *__restrict__ count_w, int32_t *__restrict__ count_b) {
  constexpr int kMaxK = kHalfkaMax + (THREATS ? kThreatMax : 0);
  __shared__ __align__(16) char s_tables[THREATS ? sizeof(EncodeTables) : 16];
  __shared__ __align__(16) int32_t s_rows[kWavesPerBlock][2 * kMaxK];
  __shared__ uint16_t s_pieces[kWavesPerBlock][2][64];
  __shared__ uint8_t s_board[kWavesPerBlock][64];
  if (THREATS) {
    const i32x4 *src = reinterpret_cast<const i32x4 *>(&kDeviceTables);
    for (int i = threadIdx.x; i < (int)(sizeof(EncodeTables) / 16); i += kBlock)
      reinterpret_cast<i32x4 *>(s_tables)[i] = src[i];
    __syncthreads();
  }
  const EncodeTables &T = *reinterpret_cast<const EncodeTables *>(s_tables);
  const int wave = uniform(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int64_t b0 = ((int64_t)blockIdx.x * kWavesPerBlock + wave) * per_wave;
  const int n = (int)std::min<int64_t>(per_wave, B - b0);  // at most 64
  const int K = enc.K;
  int32_t *rows = s_rows[wave];
  int my_pieces = 0, my_cw = 0, my_cb = 0;  // lane i's position is b0 + i
  int next = n > 0 ? boards[64 * b0 + lane] : 255;
  for (int i = 0; i < n; ++i) {  // wave-uniform
    const int pc = next;
    if (i + 1 < n) next = boards[64 * (b0 + i + 1) + lane];
    WavePosition w;
    w.occ = 0;
#pragma unroll
    for (int q = 0; q < 12; ++q) {
      w.bb[q] = ballot(pc == q);
      w.occ |= w.bb[q];
    }
    const bool occupied = pc < 12;
    const int c = pc & 1;
    w.ksq[0] = lsb64(w.bb[2 * kKing]);
    w.ksq[1] = lsb64(w.bb[2 * kKing + 1]);
    const int np = __popcll(w.occ);
    const i32x4 none = i32x4{-1, -1, -1, -1};
    for (int j = lane; j < 2 * K / 4; j += kWave) reinterpret_cast<i32x4 *>(rows)[j] = none;
    int total[2] = {0, 0}, filled[2] = {0, 0}, offset = 0;
    if (THREATS) {
      // this piece's place among its colour's, by type and then square
      int place = 0, nc[2] = {0, 0};
#pragma unroll
      for (int q = 0; q < 12; ++q) {
        if (pc == q) place = nc[q & 1] + popc_below(w.bb[q]);
        nc[q & 1] += __popcll(w.bb[q]);
      }
      w.count[0] = nc[0];
      w.count[1] = nc[1];
      w.board = s_board[wave];
      w.pieces[0] = s_pieces[wave][0];
      w.pieces[1] = s_pieces[wave][1];
      s_board[wave][lane] = (uint8_t)pc;
      if (occupied) {
        const uint16_t v = (uint16_t)(lane | pc << 8);
        s_pieces[wave][0][place + (c == 0 ? 0 : nc[0])] = v;
        s_pieces[wave][1][place + (c == 1 ? 0 : nc[1])] = v;
      }
    }
    wave_lds_barrier();
    for (int ci = 0; ci < enc.ncomp; ++ci) {
      if (enc.comp[ci] == 1) {
        if (!THREATS) continue;  // not launched so
        int found[2];
        if (np <= 32) {
          threat_rows<true>(T, w, 0, rows, K, filled[0], offset, found);
        } else {  // more pieces than a game has
          threat_rows<false>(T, w, 0, rows, K, filled[0], offset, found);
          threat_rows<false>(T, w, 1, rows, K, filled[1], offset, found);
        }
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          total[p] += found[p];
          filled[p] += min(found[p], kThreatMax);
        }
        offset += kThreatInputs;
      } else {
        // fill_halfka_feature_indices_sparse (:389-402)
        const int slot = popc_below(w.occ);
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          const int o = ((w.ksq[p] & 7) < 4 ? 7 : 0) ^ (p == 1 ? 56 : 0);
          const int kb = king_bucket(w.ksq[p] ^ o) * 768;
          if (occupied && slot < kHalfkaMax)
            rows[p * K + filled[p] + slot] = offset + (lane ^ o) + ((pc >> 1) * 2 + (c != p)) * 64 + kb;
          filled[p] += min(np, kHalfkaMax);
          total[p] += np;
        }
        offset += kHalfkaInputs;
      }
    }
    wave_lds_barrier();
    for (int j = lane; j < 2 * K / 4; j += kWave) {
      const int p = j >= K / 4 ? 1 : 0;
      i32x4 *dst = reinterpret_cast<i32x4 *>((p == 0 ? white : black) + (b0 + i) * K);
      dst[j - p * (K / 4)] = reinterpret_cast<const i32x4 *>(rows)[j];
    }
    wave_lds_barrier();  // the rows are read before the next position's fill
    if (lane == i) {
      my_pieces = np;
      my_cw = total[0];
      my_cb = total[1];
    }
  }
  if (lane >= n) return;
  const int64_t b = b0 + lane;
  if (us) us[b] = stm[b] == 0 ? 1.0f : 0.0f;
  if (psqt) psqt[b] = (my_pieces - 1) / 4;
  if (ls) ls[b] = (my_pieces - 1) / 4;
  if (count_w) count_w[b] = my_cw;
  if (count_b) count_b[b] = my_cb;
}

}  // namespace

int encode_features(const uint8_t *boards, const uint8_t *stm, int64_t B, const int32_t *comps, int ncomp,
                    int32_t *white, int32_t *black, int K, float *us, int64_t *psqt, int64_t *ls, int32_t *count_w,
                    int32_t *count_b, hipStream_t s) {
  Encoding enc{};
  enc.ncomp = ncomp;
  bool threats = false;
  for (int i = 0; i < ncomp; ++i) {
    enc.comp[i] = comps[i];
    threats = threats || comps[i] == SFT_FEATURES_THREATS;
  }
  enc.K = K;
  // positions per wave: the workgroup's table copy is shared by four times as
  // many, as long as every SIMD keeps its 8 waves
  const int64_t waves = 8 * 4 * 256;
  const int per_wave = (int)std::max<int64_t>(1, std::min<int64_t>(kWave, ceil_div(B, waves)));
  const dim3 grid((unsigned)ceil_div(B, (int64_t)per_wave * kWavesPerBlock));
  ProfScope prof(kProfEncode, s);
  hipLaunchKernelGGL((threats ? encode_kernel<true> : encode_kernel<false>), grid, dim3(kBlock), 0, s, boards, stm, B,
                     enc, per_wave, white, black, us, psqt, ls, count_w, count_b);
  return check_launch("sft_encode_features");
}

}  // namespace sft

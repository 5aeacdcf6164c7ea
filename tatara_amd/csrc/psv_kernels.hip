// PSV records -> training batch on the GPU: Huffman decode, feature-index
// extraction for the five feature sets, kingrank9 / KP-absolute progress
// buckets, score and WDL.
//
// The reference does this on CPU dataloader threads (Batch::push_decoded,
// crates/nnue-train/src/dataloader.rs:444-497, over
// ShogiBoard::from_packed_sfen, crates/shogi-format/src/packed_sfen.rs:387-449,
// and FeatureSetSpec::extract_active_features,
// crates/shogi-features/src/feature_set.rs:655-810).  Here the GPU decodes
// the 40-byte records, so the host uploads 40 bytes per position instead of
// two index rows.  Every integer result is the reference's: the emission
// order is for_each_board_piece's (BOARD_PIECE_TYPES x (black, white) x
// ascending square, packed_sfen.rs:493-540), then the two kings, then the
// hands ((black, white) x HAND_PIECE_TYPES x count).
//
// The progress bucket (ShogiProgressKPAbs::bucket_board,
// crates/shogi-features/src/progress_kpabs.rs:140-170) sums the f32 weights
// in the reference's order and evaluates exp with ref_expf(), a restatement of
// glibc's expf method (2^(k/32) table + cubic polynomial in double, the
// FMA-contracted build that glibc selects on x86-64 CPUs with FMA), which
// the reference's f32::exp calls on linux-gnu; the result equals glibc's on
// every non-NaN float.
#include "psv_kernels.hpp"

#include "common.hpp"
#include "ref_expf.hpp"

namespace tatara {

namespace {

__global__ void expf_kernel(const float* __restrict__ x, float* __restrict__ y, uint64_t n) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] = ref_expf(x[i]);
}

// ---------------------------------------------------------------------------
// pieces and BonaPiece (crates/shogi-format/src/{types,bona_piece}.rs)
// ---------------------------------------------------------------------------
constexpr int kFeHandEnd = 90, kFeOldEnd = 1548, kFKing = 1548, kEKing = 1629;

// A piece is numbered by its Huffman code, 1..7: pawn, lance, knight, silver,
// gold, bishop, rook (0: an empty square).  Its emission rank
// (BOARD_PIECE_TYPES): unpromoted id - 1, promoted pawn .. silver, horse,
// dragon 7..12.
//
// base offset [kind][is_friend] (bona_piece.rs PIECE_BASE): kinds 0..12 the
// board pieces by emission rank, 13..19 the hand pieces (13 + id - 1)
constexpr uint32_t kHandKind = 13;
__constant__ int16_t c_piece_base[20][2] = {{171, 90},   {333, 252},   {495, 414}, {657, 576}, {819, 738},
                                            {981, 900},  {1305, 1224}, {819, 738}, {819, 738}, {819, 738},
                                            {819, 738},  {1143, 1062}, {1467, 1386}, {20, 1},    {44, 39},
                                            {54, 49},    {64, 59},     {74, 69},     {82, 79},   {88, 85}};

// The Huffman id of the board code in the low bits of v (first bit lowest):
// 0; 1 0 pawn; 1 1 0 x lance / knight; 1 1 1 0 silver; 1 1 1 1 0 gold;
// 1 1 1 1 1 x bishop / rook.
__device__ __forceinline__ uint32_t board_code(uint32_t v) {
    const uint32_t n = __builtin_ctz(~v | 64u);  // leading ones, at most 6
    return n < 2 ? n : (n == 2 ? 2u + (v >> 3 & 1u) : n + 1u);
}
// code length, and the bits a square takes with promotion (not gold) and colour
__device__ __forceinline__ uint32_t code_len(uint32_t id) { return 0x66544421u >> (4 * id) & 15u; }
__device__ __forceinline__ uint32_t square_bits(uint32_t id) { return 0x88666641u >> (4 * id) & 15u; }

// A position's 256 bits, the next one lowest; zeros follow.
struct Bits {
    uint32_t w[8];
    __device__ __forceinline__ void drop(uint32_t n) {  // n < 32
#pragma unroll
        for (int k = 0; k < 7; ++k) w[k] = __builtin_amdgcn_alignbit(w[k + 1], w[k], n);
        w[7] >>= n;
    }
};

__device__ __forceinline__ int persp_sq(int sq, int persp) { return persp == 0 ? sq : 80 - sq; }
// the square with its file mirrored (squares are file * 9 + rank)
__device__ __forceinline__ int mirror_sq(int sq, bool mirror) {
    const int file = sq * 57 >> 9;  // sq / 9 for 0 <= sq <= 80
    return mirror ? 72 - 18 * file + sq : sq;
}

// ---------------------------------------------------------------------------
// A workgroup decodes kPsvRecords consecutive records.
//
//   1  wave 0, a thread per record: the Huffman code is a serial chain, walked in
//      registers (the 256 bits shift down by each code); the board pieces go
//      to LDS in square order, then the hand pieces in emission order, as
//      (kind, colour, square or count) keys
//   2  a wave per record in turn, a lane per piece: a board piece's slot in
//      emission order is the number of keys before its own (ballots over the five
//      bits of rank and colour), so a row of features is one store; with
//      progress buckets the weights are gathered into LDS in emission order
//   3  wave 0, a thread per record: the progress sum in the reference's order
//
// A record holds at most 61 pieces: a board piece takes four or more of its
// 241 bits, and with p of them the other 79 - p squares take one each and a hand
// piece three or more.  A lane per piece and king is enough.
//
// Bound by step 1's chain for few records (about 1500 dependent vector
// instructions) and by step 2's issue for many.  One thread per record for all of
// it kept boards, counters and slots in LDS and loaded the progress weights
// one after another: 65,536 records with progress buckets 132 -> 35 us,
// 1,023 without 99 -> 19 us.
// ---------------------------------------------------------------------------
constexpr int kPsvMaxActive = 40;  // the largest feature set's (halfka*: 40, halfkp: 38); a lane per slot
constexpr int kPsvRecords = 64;
constexpr int kPsvWaves = 8;
constexpr int kKeyStride = 66;     // u16 keys per record
constexpr int kProgressMax = 40;   // pieces a record's weights are gathered for (a position has 38)
constexpr int kProgressStride = 2 * kProgressMax + 1;

__global__ __launch_bounds__(kPsvWaves * 64) void psv_to_batch_kernel(PsvArgs a) {
    constexpr int R = kPsvRecords;
    __shared__ uint32_t s_rec[R * 10];
    __shared__ uint16_t s_key[R * kKeyStride];  // (kind * 2 + colour) << 7 | square (hand: count - 1)
    // flags (1 kings valid, 2 a hand past its range, 2 square maps of both sides << 2), board pieces, pieces; the
    // sides' feature bases; their two king features; the kings' progress rows
    __shared__ int32_t s_meta[R][9];
    __shared__ uint8_t s_map[4][96];  // square by (white's view, mirrored file)
    __shared__ float s_pw[R * kProgressStride];
    __shared__ int16_t s_base[40];
    const uint32_t t = threadIdx.x, lane = t % 64;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(t / 64);
    const uint32_t r0 = blockIdx.x * R;
    const uint32_t nrec = a.n - r0 < (uint32_t)R ? a.n - r0 : (uint32_t)R;
    const uint32_t* rec = reinterpret_cast<const uint32_t*>(a.psv) + (uint64_t)r0 * 10;
    for (uint32_t i = t; i < nrec * 10; i += kPsvWaves * 64) s_rec[i] = rec[i];
    if (t < 40) s_base[t] = (&c_piece_base[0][0])[t];
    if (t < 4 * 81) {
        const int m = (int)t / 81, sq = (int)t % 81;
        s_map[m][sq] = (uint8_t)mirror_sq(persp_sq(sq, m >> 1), m & 1);
    }
    __syncthreads();
    const uint32_t cap = (uint32_t)a.max_active;
    const uint32_t n_king = a.emit_king ? 2 : 0;

    // ---- 1: decode (ShogiBoard::from_packed_sfen) ----
    if (t < nrec) {
        const uint32_t* w = s_rec + t * 10;
        Bits bits;
#pragma unroll
        for (int k = 0; k < 8; ++k) bits.w[k] = w[k];
        const uint32_t tail0 = w[8], tail1 = w[9];
        const uint32_t stm = bits.w[0] & 1u, king0 = bits.w[0] >> 1 & 127u, king1 = bits.w[0] >> 8 & 127u;
        bits.drop(15);
        int cur = 15;
        uint32_t n_board = 0;
        uint16_t* keys = s_key + t * kKeyStride;
        // the coded squares: all but the kings' (a square past the board is no
        // king's square, and both kings can be on one)
        const uint32_t k_lo = king0 < king1 ? king0 : king1, k_hi = king0 < king1 ? king1 : king0;
        const uint32_t n_codes = 81u - (k_lo < 81) - (k_hi < 81 && k_hi != k_lo);
        for (uint32_t c = 0; c < n_codes;) {
            // a run of empty squares (a 0 bit each), then a piece
            uint32_t used = __builtin_ctz(bits.w[0] | 1u << 23);
            used = used < n_codes - c ? used : n_codes - c;
            c += used;
            const uint32_t v = __builtin_amdgcn_alignbit(bits.w[1], bits.w[0], used);
            if (c < n_codes && (v & 1u)) {
                const uint32_t id = board_code(v), len = square_bits(id);
                // gold has no promotion bit
                const uint32_t prom = id == 5 ? 0u : v >> code_len(id) & 1u, col = v >> (len - 1u) & 1u;
                const uint32_t rank = prom ? (id <= 4 ? id + 6 : id + 5) : id - 1;
                uint32_t sq = c + (c >= k_lo ? 1u : 0u);
                sq += k_hi != k_lo && sq >= k_hi ? 1u : 0u;
                keys[n_board++] = (uint16_t)((rank * 2 + col) << 7 | sq);
                ++c;
                used += len;
            }
            bits.drop(used);  // at most 23 + 8
            cur += (int)used;
        }
        // hands: the board code without its first (always 1) bit, a piece-box
        // bit (not gold), the owner
        uint64_t hand0 = 0, hand1 = 0;
        uint32_t n_hand = 0;
        while (cur < 256) {
            const uint32_t v = bits.w[0] << 1 | 1u;
            const uint32_t id = board_code(v);
            const uint32_t used = square_bits(id);
            const bool box = id != 5 && (v >> code_len(id) & 1u);
            const uint64_t one = box ? 0ull : 1ull << (8 * (id - 1));
            if (v >> (used - 1u) & 1u) hand1 += one;
            else hand0 += one;
            n_hand += box ? 0u : 1u;
            bits.drop(used - 1u);
            cur += (int)used - 1;
        }
        uint32_t n_piece = n_board;
        if (n_hand) {
#pragma unroll
            for (uint32_t owner = 0; owner < 2; ++owner)
#pragma unroll
                for (uint32_t hi = 0; hi < 7; ++hi) {
                    const uint32_t have = (uint32_t)((owner ? hand1 : hand0) >> (8 * hi)) & 255u;
                    for (uint32_t i = 0; i < have; ++i)
                        keys[n_piece++] = (uint16_t)(((kHandKind + hi) * 2 + owner) << 7 | i);
                }
        }
        const bool kings_ok = king0 < 81 && king1 < 81;
        if (kings_ok) {
            const int nstm = 1 - (int)stm, ks = (int)(stm ? king1 : king0), kn = (int)(stm ? king0 : king1);
            const int ki = persp_sq(ks, (int)stm), kj = persp_sq(kn, nstm);
            const bool mir_s = a.mirror && ki >= 45, mir_n = a.mirror && kj >= 45;  // files 5..8
            const int base_s = mirror_sq(ki, mir_s) * a.piece_inputs, base_n = mirror_sq(kj, mir_n) * a.piece_inputs;
            const int enemy = kEKing - (a.fold_enemy ? 81 : 0);
            s_meta[t][1] = base_s;
            s_meta[t][2] = base_n;
            s_meta[t][3] = base_s + kFKing + mirror_sq(ki, mir_s);
            s_meta[t][4] = base_s + enemy + mirror_sq(persp_sq(kn, (int)stm), mir_s);
            s_meta[t][5] = base_n + kFKing + mirror_sq(kj, mir_n);
            s_meta[t][6] = base_n + enemy + mirror_sq(persp_sq(ks, nstm), mir_n);
            s_meta[t][7] = (int)king0 * kFeOldEnd;
            s_meta[t][8] = (80 - (int)king1) * kFeOldEnd;
            // More pieces in a hand than a set has (rooks: three or more) reach past
            // the hands' range, where the reference's pack_bonapiece mirrors: a
            // hand of more than 90 - (its base as the enemy's), a byte each.
            constexpr uint64_t kPast = 0x7d776f655b5139ull;  // 127 - (70, 46, 36, 26, 16, 8, 2), pawns lowest
            const bool past = a.mirror && (((hand0 + kPast) | (hand1 + kPast)) & 0x80808080808080ull);
            s_meta[t][0] = (int)(1u | (past ? 2u : 0u) | (stm * 2 + mir_s) << 2 | (nstm * 2 + mir_n) << 4 | n_board << 8 | n_piece << 16);
        } else {
            s_meta[t][0] = 0;
        }
        const uint32_t r = r0 + t, count = kings_ok ? n_board + n_king + n_hand : 0u;
        const int8_t result = (int8_t)(tail1 >> 16 & 0xffu);
        a.nnz[r] = (int32_t)(count < cap ? count : cap);
        a.score[r] = (float)(int16_t)(tail0 & 0xffffu);
        a.wdl[r] = result > 0 ? 1.0f : (result < 0 ? 0.0f : 0.5f);
        if (a.bucket && a.bucket_mode != 2) {
            int bucket = 0;
            if (a.bucket_mode == 1) {
                // kingrank9_bucket_board: ranks from the side to move's view; the
                // u8 square arithmetic wraps as the reference's release build does
                // (only reachable with an invalid king square)
                const int flip = (uint8_t)(80 - king1);
                const int fk = stm == 0 ? (int)king0 : flip, ek = stm == 0 ? flip : (int)king0;
                bucket = (fk % 9) / 3 * 3 + (ek % 9) / 3;
            }
            a.bucket[r] = bucket;
        }
    }
    __syncthreads();

    // ---- 2: feature indices (extract_active_features) ----
    for (uint32_t rr = wave; rr < nrec; rr += kPsvWaves) {
        const uint32_t meta = __builtin_amdgcn_readfirstlane(s_meta[rr][0]);
        int32_t* so = a.stm + (uint64_t)(r0 + rr) * cap;
        int32_t* no = a.nstm + (uint64_t)(r0 + rr) * cap;
        if (!(meta & 1u)) {  // an invalid king: no features
            if (lane < cap) {
                so[lane] = -1;
                no[lane] = -1;
            }
            continue;
        }
        const uint32_t map_s = meta >> 2 & 3u, map_n = meta >> 4 & 3u, stm = map_s >> 1;
        const uint32_t n_board = meta >> 8 & 255u, n_piece = meta >> 16;
        const int base_s = s_meta[rr][1], base_n = s_meta[rr][2];

        // this lane's piece, and a board piece's slot: keys with a smaller
        // (rank, colour), or the same and a lower square (lanes are in square
        // order); the hands follow in lane order, after the kings
        const bool piece = lane < n_piece, board = lane < n_board;
        const uint32_t key = piece ? s_key[rr * kKeyStride + lane] : 0u;
        const uint32_t bin = key >> 7;
        const uint32_t sq = key & 127u, col = bin & 1u;
        uint64_t same = __ballot(board), less = 0;
#pragma unroll
        for (int b = 4; b >= 0; --b) {
            const bool one = bin >> b & 1u;
            const uint64_t ones = __ballot(board && one);
            less |= one ? same & ~ones : 0ull;
            same &= one ? ones : ~ones;
        }
        const uint32_t rank = board ? __popcll(less) + __popcll(same & ((1ull << lane) - 1ull)) : lane;
        const bool friend_s = col == stm;
        const int base_f = s_base[(bin >> 1) * 2 + 1], base_e = s_base[(bin >> 1) * 2];
        // a lane writes one slot: its piece, a king, or an empty slot
        uint32_t slot = board ? rank : lane + n_king;
        // (a hand's count goes through the identity map)
        int f_s = base_s + (friend_s ? base_f : base_e) + s_map[board ? map_s : 0u][sq];
        int f_n = base_n + (friend_s ? base_e : base_f) + s_map[board ? map_n : 0u][sq];
        if (meta & 2u) {  // a hand past the hands' range: mirrored as a board piece's square
            const int over_f = base_f + (int)sq - kFeHandEnd, over_e = base_e + (int)sq - kFeHandEnd;
            const int over_s = friend_s ? over_f : over_e, over_n = friend_s ? over_e : over_f;
            if (piece && !board && over_s >= 0) f_s = base_s + kFeHandEnd + s_map[map_s & 1u][over_s];
            if (piece && !board && over_n >= 0) f_n = base_n + kFeHandEnd + s_map[map_n & 1u][over_n];
        }
        if (!piece) {
            const uint32_t e = lane - n_piece;  // past the pieces
            const bool king = e < n_king;
            slot = king ? n_board + e : lane;  // else an empty slot
            f_s = king ? s_meta[rr][3 + (e & 1u)] : -1;
            f_n = king ? s_meta[rr][5 + (e & 1u)] : -1;
        }
        if (slot < cap) {
            so[slot] = f_s;
            no[slot] = f_n;
        }

        if (a.bucket_mode != 2) continue;
        // ---- the progress weights of every piece, in emission order ----
        float x = 0.0f, y = 0.0f;
        if (piece) {
            x = a.weights[s_meta[rr][7] + (col == 0 ? base_f : base_e) + (int)sq];
            y = a.weights[s_meta[rr][8] + (col == 1 ? base_f : base_e) + (int)(board ? 80 - sq : sq)];
        }
        float* pw = s_pw + rr * kProgressStride;
        if (n_piece <= (uint32_t)kProgressMax) {
            if (piece) {
                pw[2 * rank] = x;
                pw[2 * rank + 1] = y;
            }
        } else {
            // more pieces than a position has (arbitrary bytes): summed here
            float sum = 0.0f;
            for (uint32_t k = 0; k < n_piece; ++k) {
                const int l = (int)__builtin_ctzll(__ballot(piece && rank == k));
                sum += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), l));
                sum += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(y), l));
            }
            if (lane == 0) pw[0] = sum;
        }
    }
    if (a.bucket_mode != 2) return;
    __syncthreads();

    // ---- 3: progress bucket (BucketMode::bucket_board) ----
    if (t < nrec) {
        float sum = 0.0f;
        if (s_meta[t][0] & 1) {
            const uint32_t n_piece = (uint32_t)s_meta[t][0] >> 16;
            const float* pw = s_pw + t * kProgressStride;
            if (n_piece > (uint32_t)kProgressMax)
                sum = pw[0];
            else
                for (uint32_t k = 0; k < 2 * n_piece; ++k) sum += pw[k];
        }
        float p = 1.0f / (1.0f + ref_expf(-sum));
        p = p < 0.0f ? 0.0f : (p > 1.0f ? 1.0f : p);
        const int raw = (int)floorf(p * (float)a.num_buckets);
        if (a.bucket) a.bucket[r0 + t] = raw < 0 ? 0 : (raw > a.num_buckets - 1 ? a.num_buckets - 1 : raw);
        if (a.progress) a.progress[r0 + t] = p;
    }
}

}  // namespace

int32_t feature_set_shape(int32_t fs, FeatureSetShape& s) {
    switch (fs) {
        case 0: s = {81, 1548, 38, 0, 0, 0, 0x5D69D5B8u}; return kOk;   // halfkp
        case 1: s = {81, 1710, 40, 1, 0, 0, 0x5F134CB8u}; return kOk;   // halfka-split
        case 2: s = {81, 1629, 40, 1, 1, 0, 0xACD68C97u}; return kOk;   // halfka-merged
        case 3: s = {45, 1710, 40, 1, 0, 1, 0x2A46AC09u}; return kOk;   // halfka-hm-split
        case 4: s = {45, 1629, 40, 1, 1, 1, 0x7F134CB8u}; return kOk;   // halfka-hm-merged
        default: TATARA_REQUIRE(false, "unknown feature set");
    }
}

int32_t launch_psv_to_batch(const PsvArgs& a, hipStream_t stream) {
    TATARA_REQUIRE(a.bucket_mode >= 0 && a.bucket_mode <= 2, "unknown bucket mode");
    if (a.bucket_mode == 2) {
        TATARA_REQUIRE(a.num_buckets >= 1 && a.num_buckets <= 256, "num_buckets must be in [1, 256]");
        TATARA_REQUIRE(a.weights, "progress buckets need the KP-absolute weights");
    }
    TATARA_REQUIRE(a.max_active > 0 && a.max_active <= kPsvMaxActive && a.piece_inputs > 0, "feature set shape");
    if (a.n == 0) return kOk;
    psv_to_batch_kernel<<<ceil_div(a.n, kPsvRecords), kPsvWaves * 64, 0, stream>>>(a);
    TATARA_LAUNCHED("psv_to_batch");
    return kOk;
}

int32_t launch_expf(const float* x, float* y, uint64_t n, hipStream_t stream) {
    if (n == 0) return kOk;
    expf_kernel<<<ceil_div(n, 256), 256, 0, stream>>>(x, y, n);
    TATARA_LAUNCHED("expf");
    return kOk;
}

}  // namespace tatara

// Shared by the chunked-prefill sources (prefill_attn.hip: entry point, attention kernel,
// combine kernel; prefill_stage.h: the staging policies; prefill_flat.h: the tile loop).
//
// Rows.  The n_rep query heads of a GQA group share their kv head's keys, so a (sequence,
// kv head) pair is one attention problem of Sq x n_rep rows; row r is query r / n_rep of
// head r % n_rep.  A unit is kUnitRows rows, whatever n_rep: no wave sits on
// an absent head (with one wave per head, n_rep = 1 left three of four waves idle and
// n_rep = 7 one of eight: 512 queries of 32 heads over 4096 keys each, 158 -> 90 us with
// the repacking of the keys; 2048 queries of 28/4 heads over 4160 keys and themselves, 239
// -> 204 us).
//
// A unit pairs the u-th half-unit of 128 consecutive rows with the u-th from the end:
// waves 0-3 take the first, waves 4-7 the second, one of each on every SIMD.  With a causal
// chunk the later half sees more of it, the earlier half's waves stop computing early, and
// the others have the SIMD to themselves: the units' times differ less than with units of
// consecutive rows, which took from 66 to 97 tiles' time on the 28/4-head chunk above (204 ->
// 192 us; a tile attended by four waves takes ~0.8 of one attended by all eight).
//
// Work.  A unit's keys are tiles of 64 tokens of two kinds, each with its own staging: fp16
// (the zones' tiles, then the chunk's up to the unit's last query) and INT4.  A piece is
// 1 / pieces of a unit's tiles of one kind, one workgroup's work.  It leaves its
// online-softmax state (O relative to the row max m, m, and the row sum l, in float32) in
// its state rows, unless it is all of the unit's keys: then it writes the output.
//   kFinishOut      one kind, one piece per unit: every workgroup writes its unit's output
//   kFinishPieces   all pieces of all units, of both kinds, in one grid; the combine kernel
//                   merges their states
//   kFinishSerial   both kinds, one piece each: the fp16 kernel runs first, the INT4 kernel
//                   merges its states into its own and writes the output
// A workgroup takes one piece: with a loop over several, the tile loop's register
// allocation no longer holds (248 of 256 for INT4 tiles; all 256 for the other kinds, which
// spill 2 to 11, only kKindRefVec's loop reloading four of them).
#pragma once

#include "hkv_internal.h"

namespace hkv {

typedef _Float16 ph8 __attribute__((ext_vector_type(8)));
typedef float pf16v __attribute__((ext_vector_type(16)));
typedef float pf4 __attribute__((ext_vector_type(4)));
typedef uint32_t pu4 __attribute__((ext_vector_type(4)));
typedef uint32_t pu2 __attribute__((ext_vector_type(2)));

constexpr int kPfQ = 32;             // query rows per wave
constexpr int kPfT = 64;             // tokens per tile
constexpr float kPfLog2e = 1.4426950408889634f;
constexpr int kUnitRows = 256;       // rows per unit: 8 waves of kPfQ
constexpr int kStateFloats = 132;    // a row's state: O[128], m, l, pad
// A piece's states (kFinishPieces) in the room of 256 rows: O as [wave][16][lane] 16-byte
// pieces (piece 4 db + j of lane (n, hh): dims 32 db + 8 j + 4 hh .. +3 of row 32 wave + n),
// so that both kernels move whole kilobytes, then (m, l) per row.
constexpr int kPieceFloats = kUnitRows * kStateFloats, kPieceML = kUnitRows * kHeadDim;
// kKindRef, kKindRefVec: INT4 tiles from unpacked codes, rows of any or of 4 k tokens
enum : int { kKindF16 = 0, kKindInt4 = 1, kKindRef = 2, kKindRefVec = 3 };
// INT4 keys and values in the unpacked reference layout: one byte per code, [batch][kv
// head][int4_max_len][128], with a float scale and a byte zero point per row.
struct PfRefSource {
    const uint8_t *kc, *vc;
    const float *ks, *vs;
    const uint8_t *kz, *vz;
};

// Where the fp16 tiles of one source lie (a zone, or the causal chunk in
// the zone layout): K rows [B*Hkv][cap][128], V tiles [B*Hkv][cap/16][16 x 128].
struct PfSrc {
    const uint16_t* k;
    const uint16_t* v;
    int cap;
    int pad;
};

enum : int { kFinishOut = 0, kFinishPieces = 1, kFinishSerial = 2 };

struct PrefillParams {
    int B, Hkv, nrep, Sq;
    float scale_log2;
    int q_bf16, out_bf16;           // q / out dtype is bfloat16 (else fp16)
    const uint16_t* q;
    int64_t q_sb, q_sh, q_st;
    int has_chunk;
    int zone_max[HKV_MAX_F16_ZONES];
    const int32_t* zone_lens[HKV_MAX_F16_ZONES];
    // the fp16 sources in tile order: zones 0..2 (unused ones empty), then the chunk;
    // indexed at run time, so that no source's pointers stay in registers
    PfSrc src[HKV_MAX_F16_ZONES + 1];
    const uint8_t* pool;
    uint32_t pool_blocks;        // record counts capped at 2^31 (block ids are int32), so the
    const uint8_t* staging;      // range check is a 32-bit scalar compare; staging records are
    uint32_t staging_blocks;     // addressed by negative block ids
    int fallback_id;             // id substituted for an out-of-range one (a valid record)
    const int32_t* bt;
    int bt_stride;
    const int32_t* int4_lens;
    int int4_max_len;
    PfRefSource ref;             // the INT4 tokens of the fused entry point (no pool then)
    uint16_t* out;
    int64_t o_sb, o_sh, o_st;
    int* err;
    int units;                   // units per (sequence, kv head)
    int finish;                  // kFinish*
    int pieces[2];               // per unit, by kind (0: the launch has no tiles of the kind)
    float* state;                // state rows [.][kStateFloats]
};

// The global row of row r (< kUnitRows) of unit rb: the halves of the pairing above.  A
// middle half-unit paired with itself counts once: its second copy lies past every row.
__device__ __forceinline__ int unit_row(const PrefillParams& p, int rb, int r) {
    constexpr int kHalf = kUnitRows / 2;
    const int halves = (p.Sq * p.nrep + kHalf - 1) / kHalf;
    if (r < kHalf) return rb * kHalf + r;
    return halves - 1 - rb == rb ? halves * kHalf : (halves - 1 - rb) * kHalf + (r - kHalf);
}
// The unit's last row.
__device__ __forceinline__ int unit_last_row(const PrefillParams& p, int rb) {
    constexpr int kHalf = kUnitRows / 2;
    const int halves = (p.Sq * p.nrep + kHalf - 1) / kHalf;
    return min((halves - rb) * kHalf, p.Sq * p.nrep) - 1;
}

// The states of piece s of kind `kind` of unit `unit` (counted over all pairs).
__device__ __forceinline__ float* piece_state(const PrefillParams& p, int kind, int unit, int s) {
    const int per_unit = p.pieces[0] + p.pieces[1];
    return p.state + ((int64_t)unit * per_unit + (kind == kKindInt4 ? s : p.pieces[kKindInt4] + s)) * kPieceFloats;
}

// Tile counts of one sequence: INT4 tiles, each zone's tiles, and the causal chunk's
// tiles up to query row q_end (exclusive).
struct TileMap {
    int n4, nz_t[HKV_MAX_F16_ZONES], nc;
    int len4, lenz[HKV_MAX_F16_ZONES];
    __device__ int nf() const { return nz_t[0] + nz_t[1] + nz_t[2] + nc; }
};

__device__ __forceinline__ void make_tile_map(const PrefillParams& p, int b, int q_end, TileMap& tm) {
    tm.len4 = p.int4_lens ? min(max(load_uniform_i32(p.int4_lens, b), 0), p.int4_max_len) : p.int4_max_len;
    tm.n4 = (tm.len4 + kPfT - 1) / kPfT;
#pragma unroll
    for (int zi = 0; zi < HKV_MAX_F16_ZONES; ++zi) {
        tm.lenz[zi] = p.zone_lens[zi] ? min(max(load_uniform_i32(p.zone_lens[zi], b), 0), p.zone_max[zi]) : p.zone_max[zi];
        tm.nz_t[zi] = (tm.lenz[zi] + kPfT - 1) / kPfT;
    }
    tm.nc = p.has_chunk ? (min(q_end, p.Sq) + kPfT - 1) / kPfT : 0;
}

__device__ __forceinline__ uint32_t pack2(float a, float b) {
    return (uint32_t)f2h_rn(a) | ((uint32_t)f2h_rn(b) << 16);
}
__device__ __forceinline__ uint32_t pack2bf(float a, float b) {
    return (uint32_t)f2bf_rn(a) | ((uint32_t)f2bf_rn(b) << 16);
}

// Eight bf16 values to fp16: exact in [2^-14, 65504]; `over` is set when a finite
// value leaves the fp16 range (it becomes +-inf).
__device__ __forceinline__ pu4 bf16x8_to_f16(pu4 w, bool& over) {
    pu4 r;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float lo = __uint_as_float(w[e] << 16), hi = __uint_as_float(w[e] & 0xffff0000u);
        const uint32_t a = f2h_rn(lo), b = f2h_rn(hi);
        over |= (((a & 0x7fffu) == 0x7c00u) && fabsf(lo) < INFINITY) ||
                (((b & 0x7fffu) == 0x7c00u) && fabsf(hi) < INFINITY);
        r[e] = a | (b << 16);
    }
    return r;
}

// Four output dims at `op`: x times inv, rounded to the output dtype.
__device__ __forceinline__ void store_out4(const PrefillParams& p, uint16_t* op, pf4 x, float inv) {
    *(pu2*)op = p.out_bf16 ? pu2{pack2bf(x[0] * inv, x[1] * inv), pack2bf(x[2] * inv, x[3] * inv)}
                           : pu2{pack2(x[0] * inv, x[1] * inv), pack2(x[2] * inv, x[3] * inv)};
}

// Writes this lane's final output: acc[db][4j + i] is O^T[dim 32db + 8j + 4hh + i][its
// row], l the row's softmax sum.
__device__ __forceinline__ void write_out(const PrefillParams& p, int b, int qh, int qrow, int hh,
                                          const pf16v (&acc)[4], float l) {
    const float inv = l > 0.f ? 1.0f / l : 0.f;
    uint16_t* op = p.out + (int64_t)b * p.o_sb + (int64_t)qh * p.o_sh + (int64_t)qrow * p.o_st;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int j = 0; j < 4; ++j)
            store_out4(p, op + 32 * db + 8 * j + 4 * hh,
                       pf4{acc[db][4 * j + 0], acc[db][4 * j + 1], acc[db][4 * j + 2], acc[db][4 * j + 3]}, inv);
}

}  // namespace hkv

// Chunked-prefill attention over [fp16 zones | causal chunk | INT4 pool] on MFMA: the
// entry point, the attention kernel and the combine kernel (tile loop: prefill_flat.h;
// staging: prefill_stage.h; rows, units and the work plan: prefill_common.h).
//
// Math (fused_dequant_attn.py:242-247,385-390; kernels/fused_dequant_attn.py:371-435
// is the reference entry point): out[q] = softmax_t(q . K_t * sm_scale) V_t over every
// INT4 token (dequantized as (code - zero point) x scale), every fp16 zone token and the
// chunk's own tokens t <= q (causal), GQA q head i -> kv head i / n_rep.
//
// INT4 tiles are staged into LDS as fp16 K rows (code - zero point) x K scale and V^T
// rows (code - zero point) x V scale; the queries carry sm_scale x log2 e (rounded to
// fp16 once), so the scores come out of the MFMAs in the log2 domain.  The staging rounds
// the scale to fp16 and then the product: two roundings, within about 1.5 fp16 ulps of
// the Path C dequantization's one while the scale is at least 2^-14 (store_k4 / store_v4).
// The chunk's K/V are first rewritten in the zone layout (zone_write_kernel).
#include "prefill_stage.h"

#include <algorithm>
#include <cmath>

namespace hkv {
namespace {

template <int kKind, int kTeam>
using Stage = typename std::conditional<
    kKind == kKindF16, F16Stage<kTeam>,
    typename std::conditional<kKind == kKindInt4, Int4Stage<kTeam>, RefStage<kTeam, kKind == kKindRefVec>>::type>::type;

// Writes a piece's result: a state, or the output (with kFinishSerial, of the fp16
// kernel's states and this one's).
template <int kKind>
__device__ __forceinline__ void finish(const PrefillParams& p, const TileMap& tm, int bh, int rb, int s, int tid,
                                       pf16v (&acc)[4], float m, float l) {
    const int hh = (tid >> 5) & 1, r0 = (tid >> 6) * kPfQ + (tid & 31);   // row of the unit
    const int row = unit_row(p, rb, r0);
    if (row >= p.Sq * p.nrep) return;
    const int wave = tid >> 6;
    if (p.finish == kFinishPieces) {
        float* st = piece_state(p, kKind, bh * p.units + rb, s);
        pf4* o = (pf4*)st + (wave * 16) * 64 + (tid & 63);
#pragma unroll
        for (int db = 0; db < 4; ++db)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                o[(4 * db + j) * 64] = pf4{acc[db][4 * j + 0], acc[db][4 * j + 1], acc[db][4 * j + 2], acc[db][4 * j + 3]};
        if (hh == 0) *(float2*)(st + kPieceML + 2 * r0) = make_float2(m, l);
        return;
    }
    const int64_t own_row = (int64_t)bh * (p.Sq * p.nrep) + row;   // kFinishSerial
    if (kKind == kKindF16 && p.finish == kFinishSerial && tm.n4 > 0) {
        float* st = p.state + own_row * kStateFloats;
#pragma unroll
        for (int db = 0; db < 4; ++db)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                *(pf4*)(st + 32 * db + 8 * j + 4 * hh) =
                    pf4{acc[db][4 * j + 0], acc[db][4 * j + 1], acc[db][4 * j + 2], acc[db][4 * j + 3]};
        if (hh == 0) *(float2*)(st + kHeadDim) = make_float2(m, l);
        return;
    }
    if (kKind == kKindInt4 && p.finish == kFinishSerial && tm.nf() > 0) {
        // merge the fp16 kernel's state of this row with this kernel's: rescale both to
        // the common max
        const float* st = p.state + own_row * kStateFloats;
        const float2 z = *(const float2*)(st + kHeadDim);
        const float mn = fmaxf(m, z.x);
        const float fa = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - mn);
        const float fz = z.x == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(z.x - mn);
#pragma unroll
        for (int db = 0; db < 4; ++db)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const f4 oz = *(const f4*)(st + 32 * db + 8 * j + 4 * hh);
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[db][4 * j + i] = acc[db][4 * j + i] * fa + oz[i] * fz;
            }
        l = l * fa + z.y * fz;
    }
    const int b = bh / p.Hkv, h = bh - b * p.Hkv;
    write_out(p, b, h * p.nrep + row % p.nrep, row / p.nrep, hh, acc, l);
}

// Workgroup wg of kind kKind.
template <int kKind>
__device__ __forceinline__ void attend(const PrefillParams& p, int wg, uint8_t* lds) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int team = wave >> 2, wt = wave & 3;
    const int n = lane & 31, hh = lane >> 5;
    const int BH = p.B * p.Hkv;
    // Dispatch goes round-robin over the 8 XCDs by workgroup id: with the pairs innermost,
    // the workgroups of one pair run on one XCD and share its L2 when the pairs are a
    // multiple of 8.  The first units, with the most chunk tiles, come first.
    const int bh = wg % BH;
    const int rb = wg / BH % p.units;
    constexpr int kPlan = kKind == kKindF16 ? kKindF16 : kKindInt4;   // unpacked codes are INT4 tiles
    const int s = wg / BH / p.units, ns = p.pieces[kPlan];
    const int b = bh / p.Hkv, h = bh - b * p.Hkv;
    const int row0 = unit_row(p, rb, wave * kPfQ);   // this wave's first row
    TileMap tm;
    make_tile_map(p, b, unit_last_row(p, rb) / p.nrep + 1, tm);
    const int tiles = kKind == kKindF16 ? tm.nf() : tm.n4;
    // both kinds, one after the other: the other kernel finishes a sequence without tiles
    // of this kind
    if (p.finish == kFinishSerial && tiles == 0 && (kKind != kKindF16 || tm.n4 > 0)) return;
    // pieces start at multiples of the loop's round of kFlatBufs tiles
    const int rounds = (tiles + kFlatBufs - 1) / kFlatBufs;
    const int t0 = rounds * s / ns * kFlatBufs, t1 = min(tiles, rounds * (s + 1) / ns * kFlatBufs);
    const int T = (t1 - t0 + kFlatBufs - 1) / kFlatBufs * kFlatBufs;
    // of these, a wave attends those up to its last query's
    int Tc = row0 < p.Sq * p.nrep ? T : 0;
    const int q_hi = min((row0 + kPfQ - 1) / p.nrep, p.Sq - 1);
    if (kKind == kKindF16 && tm.nc > 0 && Tc > 0) {
        const int last = tm.nf() - tm.nc + q_hi / kPfT;
        Tc = min(T, max(0, last - t0 + kFlatBufs) / kFlatBufs * kFlatBufs);
    }

    ph8 qf[8];
    const int qrow = min((row0 + n) / p.nrep, p.Sq - 1);
    flat_load_q(p,
                p.q + (int64_t)b * p.q_sb + (int64_t)(h * p.nrep + (row0 + n) % p.nrep) * p.q_sh + (int64_t)qrow * p.q_st,
                row0 + n < p.Sq * p.nrep, hh, qf);
    pf16v acc[4];
    float m = -INFINITY, l = 0.f;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[db][r] = 0.f;
    if (kKind == kKindF16) {   // read behind the loop's first barrier
        for (int i = threadIdx.x; i < kZeroBytes / 16; i += kFlatThreads) ((pu4*)(lds + kFlatLdsBytes))[i] = pu4{0u, 0u, 0u, 0u};
    }
    const FlatWave fw{b, h, wt, lane, n, hh, qrow, row0 / p.nrep, q_hi};
    if (T > 0) {
        if (team == 0) {
            Stage<kKind, 0> pol(p, tm, fw, t0, t1);
            flat_tiles(pol, tm, fw, lds, qf, acc, m, l, Tc, T);
        } else {
            // waves 4-7 (the V^T staging, the larger share of VALU work) win issue ties
            // against the older waves 0-3 on their SIMDs
            __builtin_amdgcn_s_setprio(1);
            Stage<kKind, 1> pol(p, tm, fw, t0, t1);
            flat_tiles(pol, tm, fw, lds, qf, acc, m, l, Tc, T);
            __builtin_amdgcn_s_setprio(0);
        }
    }
    l += __shfl_xor(l, 32);
    // from here on the lane's row is worked out again (from an opaque thread index), so that
    // nothing of it lives in registers across the tile loop
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    finish<kPlan>(p, tm, bh, rb, s, tid, acc, m, l);
}

// One workgroup per CU: 8 waves (two per SIMD), up to 256 registers per wave.  kKinds: a bit
// per kind of tiles in the grid.  A kernel for each set of kinds: with both kinds' loops in
// every kernel, 12 registers spilled and 2048 queries over 131K INT4 keys took 4.37 ms, not
// 4.27 (same box).
template <int kKinds>
__global__ __launch_bounds__(kFlatThreads, 1) void prefill_attn_kernel(PrefillParams p) {
    touch_kernel_args(p);
    extern __shared__ __align__(16) uint8_t lds_raw[];
    constexpr int kF16 = 1 << kKindF16, kInt4 = 1 << kKindInt4;
    if constexpr (kKinds == kF16) {
        attend<kKindF16>(p, blockIdx.x, lds_raw);
    } else if constexpr (kKinds == kInt4) {
        attend<kKindInt4>(p, blockIdx.x, lds_raw);
    } else if constexpr (kKinds == 1 << kKindRef) {
        attend<kKindRef>(p, blockIdx.x, lds_raw);
    } else if constexpr (kKinds == 1 << kKindRefVec) {
        attend<kKindRefVec>(p, blockIdx.x, lds_raw);
    } else {
        const int n4 = p.B * p.Hkv * p.units * p.pieces[kKindInt4];
        if ((int)blockIdx.x < n4) attend<kKindInt4>(p, blockIdx.x, lds_raw);
        else attend<kKindF16>(p, (int)blockIdx.x - n4, lds_raw);
    }
}

// Merges the states of a unit's pieces (kFinishPieces).  One workgroup per 32 rows of a
// unit (a wave's), wave db over dims 32 db .. +31, with the attention kernel's lane layout.
// Bound by the reads of the states (520 B per row and piece), which the Infinity Cache
// mostly serves: 256 pieces, 33 MB, in 7.8 us (11.7 us with row-major states, whose 16-byte
// pieces of a wave's store lie in 32 rows).
__global__ __launch_bounds__(256) void prefill_combine_kernel(PrefillParams p) {
    touch_kernel_args(p);
    const int unit = (int)blockIdx.x >> 3, wave = (int)blockIdx.x & 7;
    const int bh = unit / p.units, rb = unit - bh * p.units;
    const int lane = threadIdx.x & 63, db = threadIdx.x >> 6, n = lane & 31, hh = lane >> 5;
    const int row = unit_row(p, rb, wave * kPfQ + n);
    if (__ballot(row < p.Sq * p.nrep) == 0) return;
    const int np = p.pieces[0] + p.pieces[1];
    const float* st = p.state + (int64_t)unit * np * kPieceFloats;
    const int ml = kPieceML + 2 * (wave * kPfQ + n), oo = ((wave * 16 + 4 * db) * 64 + lane) * 4;
    float M = -INFINITY;
#pragma unroll 4
    for (int i = 0; i < np; ++i) M = fmaxf(M, st[(int64_t)i * kPieceFloats + ml]);
    pf4 O[4] = {};
    float L = 0.f;
#pragma unroll 4
    for (int i = 0; i < np; ++i) {
        const float* s = st + (int64_t)i * kPieceFloats;
        const float2 x = *(const float2*)(s + ml);
        const float e = x.x == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(x.x - M);
        L += x.y * e;
#pragma unroll
        for (int j = 0; j < 4; ++j) O[j] += *(const pf4*)(s + oo + j * 256) * e;
    }
    if (row >= p.Sq * p.nrep) return;
    const int b = bh / p.Hkv, h = bh - b * p.Hkv;
    uint16_t* op = p.out + (int64_t)b * p.o_sb + (int64_t)(h * p.nrep + row % p.nrep) * p.o_sh +
                   (int64_t)(row / p.nrep) * p.o_st;
    const float inv = L > 0.f ? 1.0f / L : 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) store_out4(p, op + 32 * db + 8 * j + 4 * hh, O[j], inv);
}

// ---- the work plan (host)
int num_cus() {
    static std::atomic<int> cached[64];   // per device (partition modes can differ)
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 256;
    const int c = cached[dev & 63].load(std::memory_order_relaxed);
    if (c > 0) return c;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) return 256;
    cached[dev & 63].store(n, std::memory_order_relaxed);
    return n;
}

// Why split: 203 queries of 32/8 heads are 32 units on 256 CUs; over 32,960 keys they took
// 945 us unsplit and 155 us in 8 pieces each (7 INT4, 1 fp16).  Why not always: every piece
// writes and reads 135 KB of states, 16 us for 256 pieces; 256 equal units gain nothing.
// Pieces hold whole rounds of the loop (64 pieces for 18 tiles cost 98 us, 6 pieces 32 us).
// What the schedules cost, in INT4 tiles of one workgroup (~2 us each).  Workgroups run
// longest first, one per CU, so CU round k ends with workgroup k x CUs of that order.
constexpr double kF16Tile = 1.03;      // an fp16 tile (4x the K/V bytes of an INT4 one)
constexpr double kSegTiles = 1.5;      // pipeline start and end of one tile loop
constexpr double kLaunchTiles = 2.0;   // one more launch in the stream
constexpr double kPieceTiles = 0.03;   // one piece's states: 135 KB written and read at ~4 TB/s
constexpr int kMaxPieces = 64;

struct Plan {
    int units, finish, pieces[2];
    int64_t state_rows;
};

// Time of `n4` INT4 workgroups of len4 tiles each beside `nf` fp16 ones of lenf tiles.
double grid_tiles(int cus, int64_t n4, double len4, int64_t nf, double lenf) {
    double t = 0;
    for (int64_t r = 0; r < n4 + nf; r += cus) t += kSegTiles + ((len4 >= lenf) == (r < (len4 >= lenf ? n4 : nf)) ? len4 : lenf);
    return t;
}

// The schedule of a launch over tiles[kind] tiles per sequence (by the maximal lengths)
// plus, with `chunk`, the causal chunk's, that needs at most max_rows state rows.
Plan make_plan(int64_t bh, int nrep, int sq, const int64_t (&tiles)[2], bool chunk, int64_t max_rows) {
    Plan best;
    best.units = (int)(((int64_t)sq * nrep + kUnitRows - 1) / kUnitRows);
    const int64_t all = bh * best.units;
    const int cus = num_cus();
    const bool has4 = tiles[kKindInt4] > 0, hasf = tiles[kKindF16] > 0 || chunk || !has4, both = has4 && hasf;
    // the pairing of the rows evens out the chunk's tiles: about the middle row's per unit
    const double len4 = (double)tiles[kKindInt4];
    const double lenf = ((double)tiles[kKindF16] + (chunk ? 0.55 * sq / kPfT + 1 : 0)) * kF16Tile;
    best.pieces[kKindF16] = hasf;
    best.pieces[kKindInt4] = has4;
    best.finish = both ? kFinishSerial : kFinishOut;
    best.state_rows = both ? bh * sq * nrep : 0;
    // Many units per CU even out by themselves, and their states would take gigabytes.
    if (all > 2 * cus) return best;
    double t_best = both ? kLaunchTiles : 0;
    if (has4) t_best += grid_tiles(cus, all, std::ceil(len4 / kFlatBufs) * kFlatBufs, 0, 0);
    if (hasf) t_best += grid_tiles(cus, 0, 0, all, lenf);
    // pieces of up to `len` tiles of either kind, in the loop's rounds
    for (int len = kFlatBufs; len <= 1024; len += std::max(kFlatBufs, len / 64 * kFlatBufs)) {
        const auto pieces = [&](double tiles_k) { return (int)std::min<double>(kMaxPieces, std::ceil(tiles_k / len)); };
        const int p4 = has4 ? pieces(len4) : 0, pf = hasf ? pieces(lenf) : 0;
        const int64_t n = all * (p4 + pf);
        if (p4 + pf < 2 || n > 4 * cus || n * kUnitRows > max_rows) continue;
        const auto longest = [](double tiles_k, int np) { return np ? std::ceil(std::ceil(tiles_k / kFlatBufs) / np) * kFlatBufs : 0; };
        const double t = grid_tiles(cus, all * p4, longest(len4, p4), all * pf, longest(lenf, pf)) + kLaunchTiles +
                         (double)n * kPieceTiles;
        if (t < t_best) {
            t_best = t;
            best.finish = kFinishPieces;
            best.pieces[kKindInt4] = p4;
            best.pieces[kKindF16] = pf;
            best.state_rows = n * kUnitRows;
        }
    }
    return best;
}

Plan plan_of(const HkvPrefillArgs* a, int64_t max_rows) {
    int64_t tiles[2] = {0, ((int64_t)a->int4_max_len + kPfT - 1) / kPfT};
    for (int i = 0; i < a->num_f16_zones; ++i) tiles[kKindF16] += ((int64_t)a->f16[i].max_len + kPfT - 1) / kPfT;
    return make_plan((int64_t)a->batch * a->num_kv_heads, a->num_q_heads / a->num_kv_heads, a->num_queries, tiles,
                     a->chunk_k != nullptr, max_rows);
}
// Workspace bytes of the chunk in the zone layout (K rows, then V tiles).
size_t chunk_ws_bytes(const HkvPrefillArgs* a) {
    if (!a->chunk_k) return 0;
    const size_t ccap = ((size_t)a->num_queries + kBlockTokens - 1) / kBlockTokens * kBlockTokens;
    return 2 * (size_t)a->batch * a->num_kv_heads * ccap * kHeadDim * 2;
}

// Sequences b0 .. b0 + n - 1 of a launch.  The state rows are used again by every slice: the
// stream orders a slice's kernels after those of the one before.
PrefillParams batch_slice(const PrefillParams& p, int b0, int n) {
    PrefillParams s = p;
    const int64_t pairs = (int64_t)b0 * p.Hkv, codes = pairs * p.int4_max_len;
    s.B = n;
    s.q += b0 * p.q_sb;
    s.out += b0 * p.o_sb;
    for (const int32_t*& l : s.zone_lens)
        if (l) l += b0;
    for (PfSrc& f : s.src)
        if (f.k) {
            f.k += pairs * f.cap * kHeadDim;
            f.v += pairs * f.cap * kHeadDim;
        }
    if (s.bt) s.bt += (int64_t)b0 * p.bt_stride;
    if (s.int4_lens) s.int4_lens += b0;
    if (s.ref.kc) {
        s.ref.kc += codes * kHeadDim;
        s.ref.vc += codes * kHeadDim;
        s.ref.ks += codes;
        s.ref.vs += codes;
        s.ref.kz += codes;
        s.ref.vz += codes;
    }
    return s;
}

int launch_slice(PrefillParams& p, const Plan& pl, bool ref, hipStream_t stream) {
    static void (*const fns[9])(PrefillParams) = {
        nullptr, prefill_attn_kernel<1>, prefill_attn_kernel<2>, prefill_attn_kernel<3>, prefill_attn_kernel<4>,
        nullptr, nullptr, nullptr, prefill_attn_kernel<8>};
    static std::atomic<uint64_t> raised[9];   // four tile buffers exceed the 64 KB default
    const unsigned all = (unsigned)(p.B * p.Hkv * p.units);
    const bool serial = pl.finish == kFinishSerial;
    for (int kind = 0; kind < (serial ? 2 : 1); ++kind) {
        int kinds = 0;
        for (int k = 0; k < 2; ++k) {
            p.pieces[k] = serial && k != kind ? 0 : pl.pieces[k];
            if (p.pieces[k] > 0) kinds |= 1 << k;
        }
        if (ref) kinds = 1 << (p.int4_max_len % 4 == 0 ? kKindRefVec : kKindRef);
        const int lds = kFlatLdsBytes + (kinds & (1 << kKindF16) ? kZeroBytes : 0);
        HKV_RAISE_LDS(fns[kinds], lds, raised[kinds]);
        hipLaunchKernelGGL(fns[kinds], dim3(all * (unsigned)(p.pieces[0] + p.pieces[1])), dim3(kFlatThreads), lds, stream,
                           p);
        HKV_LAUNCH_CHECK("prefill_attn_kernel");
    }
    if (pl.finish == kFinishPieces) {
        hipLaunchKernelGGL(prefill_combine_kernel, dim3(all * kFlatWaves), dim3(256), 0, stream, p);
        HKV_LAUNCH_CHECK("prefill_combine_kernel");
    }
    return HKV_OK;
}

// The pairs and units are all in the grid's x, which takes fewer than 2^32 threads: a call
// with more goes by slices of its sequences (it has too many units to be split into pieces).
constexpr int64_t kMaxGridUnits = ((1ll << 32) - 1) / kFlatThreads;

int launch_attn(PrefillParams& p, const Plan& pl, bool ref, hipStream_t stream) {
    p.units = pl.units;
    p.finish = pl.finish;
    const int64_t per_seq = (int64_t)p.Hkv * p.units;
    if (p.B * per_seq <= kMaxGridUnits) return launch_slice(p, pl, ref, stream);
    const int step = (int)std::max<int64_t>(1, kMaxGridUnits / per_seq);
    for (int b0 = 0; b0 < p.B; b0 += step) {
        PrefillParams s = batch_slice(p, b0, std::min(step, p.B - b0));
        const int rc = launch_slice(s, pl, ref, stream);
        if (rc != HKV_OK) return rc;
    }
    return HKV_OK;
}

}  // namespace
}  // namespace hkv

using namespace hkv;

// The launch behind both entry points; `ref` is null, or holds the INT4 tokens in place of
// the pool.
static int prefill_launch(const HkvPrefillArgs* a, const PfRefSource* ref, void* stream) {
    HKV_REQUIRE(a != nullptr, HKV_ERR_ARG, "hkv_prefill_attn: null args");
    HKV_REQUIRE(a->head_dim == kHeadDim, HKV_ERR_UNSUPPORTED, "hkv_prefill_attn: head_dim %d != 128", a->head_dim);
    HKV_REQUIRE(a->batch > 0 && a->num_kv_heads > 0 && a->num_q_heads > 0 && a->num_queries > 0, HKV_ERR_ARG,
                "hkv_prefill_attn: bad sizes");
    HKV_REQUIRE(a->num_q_heads % a->num_kv_heads == 0, HKV_ERR_ARG,
                "hkv_prefill_attn: num_q_heads %d not a multiple of num_kv_heads %d", a->num_q_heads,
                a->num_kv_heads);
    HKV_REQUIRE(a->num_f16_zones >= 0 && a->num_f16_zones <= HKV_MAX_F16_ZONES, HKV_ERR_ARG,
                "hkv_prefill_attn: num_f16_zones out of range");
    HKV_REQUIRE(a->q && a->out, HKV_ERR_ARG, "hkv_prefill_attn: null q/out");
    HKV_REQUIRE((a->q_dtype == HKV_DTYPE_F16 || a->q_dtype == HKV_DTYPE_BF16) &&
                    (a->chunk_dtype == HKV_DTYPE_F16 || a->chunk_dtype == HKV_DTYPE_BF16) &&
                    (a->out_dtype == HKV_DTYPE_F16 || a->out_dtype == HKV_DTYPE_BF16),
                HKV_ERR_ARG, "hkv_prefill_attn: q/chunk/out dtype must be fp16 or bf16");
    HKV_REQUIRE((((uintptr_t)a->q) & 15) == 0 && a->q_stride_b % 8 == 0 && a->q_stride_h % 8 == 0 &&
                    a->q_stride_t % 8 == 0,
                HKV_ERR_ARG, "hkv_prefill_attn: q must be 16-byte aligned with strides multiple of 8");
    HKV_REQUIRE((((uintptr_t)a->out) & 7) == 0 && a->out_stride_b % 4 == 0 && a->out_stride_h % 4 == 0 &&
                    a->out_stride_t % 4 == 0,
                HKV_ERR_ARG, "hkv_prefill_attn: out must be 8-byte aligned with strides multiple of 4");
    if (a->chunk_k || a->chunk_v) {
        HKV_REQUIRE(a->chunk_k && a->chunk_v, HKV_ERR_ARG, "hkv_prefill_attn: chunk K and V must both be given");
        HKV_REQUIRE((((uintptr_t)a->chunk_k | (uintptr_t)a->chunk_v) & 15) == 0 && a->chunk_stride_b % 8 == 0 &&
                        a->chunk_stride_h % 8 == 0 && a->chunk_stride_t % 8 == 0,
                    HKV_ERR_ARG, "hkv_prefill_attn: chunk K/V must be 16-byte aligned, strides multiple of 8");
    }
    HKV_REQUIRE(a->int4_max_len >= 0, HKV_ERR_ARG, "hkv_prefill_attn: int4_max_len < 0");
    if (a->int4_max_len > 0 && !ref) {
        HKV_REQUIRE(a->block_table && ((a->pool && a->pool_blocks > 0) || (a->staging && a->staging_blocks > 0)),
                    HKV_ERR_ARG, "hkv_prefill_attn: INT4 zone without pool/staging records or block table");
        HKV_REQUIRE(a->pool_blocks >= 0 && a->staging_blocks >= 0 && a->staging_blocks <= (1ll << 31),
                    HKV_ERR_ARG, "hkv_prefill_attn: bad pool/staging block counts");
        HKV_REQUIRE((((uintptr_t)a->pool | (uintptr_t)a->staging) & 15) == 0, HKV_ERR_ARG,
                    "hkv_prefill_attn: pool/staging must be 16-byte aligned");
        HKV_REQUIRE((int64_t)a->bt_stride * kBlockTokens >= a->int4_max_len, HKV_ERR_CAPACITY,
                    "hkv_prefill_attn: block table stride too small");
    }
    for (int i = 0; i < a->num_f16_zones; ++i) {
        const HkvF16Zone& z = a->f16[i];
        HKV_REQUIRE(z.max_len >= 0 && z.max_len <= z.capacity && z.capacity % kBlockTokens == 0, HKV_ERR_ARG,
                    "hkv_prefill_attn: zone %d length/capacity invalid", i);
        if (z.max_len > 0)
            HKV_REQUIRE(z.k && z.v && (((uintptr_t)z.k | (uintptr_t)z.v) & 15) == 0, HKV_ERR_ARG,
                        "hkv_prefill_attn: zone %d k/v null or misaligned", i);
    }
    const int nrep = a->num_q_heads / a->num_kv_heads;
    const int ngrp = (nrep + 3) / 4;
    // the kernel's linear workgroup id (pair, unit) is a 32-bit int: at most one unit per 64
    // queries and four heads of a group
    const int64_t qblocks = ((int64_t)a->num_queries + 63) / 64;
    HKV_REQUIRE((int64_t)a->num_kv_heads * ngrp < 65536 && a->batch < 65536 &&
                    qblocks * a->num_kv_heads * ngrp < (1ll << 31),
                HKV_ERR_ARG, "hkv_prefill_attn: grid too large");
    PrefillParams p;
    p.B = a->batch;
    p.Hkv = a->num_kv_heads;
    p.nrep = nrep;
    p.Sq = a->num_queries;
    p.scale_log2 = a->sm_scale * kPfLog2e;
    p.q_bf16 = a->q_dtype == HKV_DTYPE_BF16;
    p.out_bf16 = a->out_dtype == HKV_DTYPE_BF16;
    p.q = a->q;
    p.q_sb = a->q_stride_b;
    p.q_sh = a->q_stride_h;
    p.q_st = a->q_stride_t;
    for (int i = 0; i < HKV_MAX_F16_ZONES; ++i) {
        const bool on = i < a->num_f16_zones;
        p.zone_max[i] = on ? a->f16[i].max_len : 0;
        p.zone_lens[i] = on ? a->f16[i].lens : nullptr;
        p.src[i] = on && a->f16[i].k ? PfSrc{a->f16[i].k, a->f16[i].v, a->f16[i].capacity, 0} : PfSrc{nullptr, nullptr, 16, 0};
    }
    p.src[HKV_MAX_F16_ZONES] = PfSrc{nullptr, nullptr, 16, 0};
    p.has_chunk = a->chunk_k != nullptr;
    p.pool = a->pool;
    p.pool_blocks = a->pool ? (uint32_t)std::min<int64_t>(a->pool_blocks, 1ll << 31) : 0u;
    p.staging = a->staging;
    p.staging_blocks = a->staging ? (uint32_t)std::min<int64_t>(a->staging_blocks, 1ll << 31) : 0u;
    p.fallback_id = p.pool_blocks > 0 ? 0 : -1;
    p.bt = a->block_table;
    p.bt_stride = a->bt_stride;
    p.int4_lens = a->int4_lens;
    p.int4_max_len = a->int4_max_len;
    p.ref = ref ? *ref : PfRefSource{};
    p.out = a->out;
    p.o_sb = a->out_stride_b;
    p.o_sh = a->out_stride_h;
    p.o_st = a->out_stride_t;
    p.err = a->err_flag;
    // The workspace: the chunk's K/V in the zone layout, written by the zone writer before
    // the attention kernel runs, then the state rows.  A split launch takes more of those
    // than the documented size has room for; without them it runs unsplit.
    bool zone_keys = a->chunk_k != nullptr;
    for (int i = 0; i < a->num_f16_zones; ++i) zone_keys = zone_keys || a->f16[i].max_len > 0;
    const bool ws_ok = a->workspace != nullptr && (((uintptr_t)a->workspace) & 15) == 0;
    if (a->chunk_k != nullptr || (zone_keys && a->int4_max_len > 0)) {
        const size_t need = hkv_prefill_workspace_bytes(a->batch, a->num_q_heads, a->num_queries);
        HKV_REQUIRE(ws_ok && a->workspace_bytes >= need, HKV_ERR_ARG,
                    "hkv_prefill_attn: a causal chunk, or INT4 and zone keys, need a 16-byte aligned "
                    "workspace of %zu bytes (hkv_prefill_workspace_bytes), got %zu", need,
                    a->workspace ? a->workspace_bytes : 0);
    }
    uint8_t* ws = (uint8_t*)a->workspace;
    const size_t chunk_bytes = chunk_ws_bytes(a);
    p.state = (float*)(ws + chunk_bytes);
    if (a->chunk_k != nullptr) {
        const int ccap = (a->num_queries + kBlockTokens - 1) / kBlockTokens * kBlockTokens;
        p.src[HKV_MAX_F16_ZONES] = PfSrc{(const uint16_t*)ws, (const uint16_t*)(ws + chunk_bytes / 2), ccap, 0};
        HkvZoneWriteArgs zw = {};
        zw.k = a->chunk_k;
        zw.v = a->chunk_v;
        zw.src_stride_b = a->chunk_stride_b;
        zw.src_stride_h = a->chunk_stride_h;
        zw.src_stride_t = a->chunk_stride_t;
        zw.batch = a->batch;
        zw.num_kv_heads = a->num_kv_heads;
        zw.head_dim = kHeadDim;
        zw.num_tokens = a->num_queries;
        zw.slot_start = nullptr;
        zw.capacity = ccap;
        zw.ring = 0;
        zw.zone_k = (uint16_t*)ws;
        zw.zone_v = (uint16_t*)(ws + chunk_bytes / 2);
        zw.slot_base = 0;
        zw.dtype = a->chunk_dtype;
        zw.err_flag = a->err_flag;
        const int rc = hkv_zone_write(&zw, stream);
        if (rc != HKV_OK) return rc;
    }
    const int64_t rows = ws_ok && a->workspace_bytes > chunk_bytes
                             ? (int64_t)((a->workspace_bytes - chunk_bytes) / (kStateFloats * sizeof(float)))
                             : 0;
    return launch_attn(p, plan_of(a, rows), ref != nullptr, (hipStream_t)stream);
}

extern "C" int hkv_prefill_attn(const HkvPrefillArgs* a, void* stream) {
    clear_error();
    return prefill_launch(a, nullptr, stream);
}

// The prefill call that a fused forward makes: its INT4 tokens are all its keys.
static HkvPrefillArgs fused_as_prefill(const HkvFusedArgs* f) {
    HkvPrefillArgs a = {};
    a.batch = f->batch;
    a.num_q_heads = f->num_q_heads;
    a.num_kv_heads = f->num_kv_heads;
    a.head_dim = f->head_dim;
    a.num_queries = f->num_queries;
    a.sm_scale = f->sm_scale;
    a.q = f->q;
    a.q_stride_b = f->q_stride_b;
    a.q_stride_h = f->q_stride_h;
    a.q_stride_t = f->q_stride_t;
    a.int4_max_len = f->num_tokens;
    a.out = f->out;
    a.out_stride_b = f->out_stride_b;
    a.out_stride_h = f->out_stride_h;
    a.out_stride_t = f->out_stride_t;
    a.err_flag = f->err_flag;
    a.q_dtype = f->q_dtype;
    a.out_dtype = f->out_dtype;
    a.workspace = f->workspace;
    a.workspace_bytes = f->workspace_bytes;
    return a;
}

extern "C" int hkv_fused_forward(const HkvFusedArgs* f, void* stream) {
    clear_error();
    HKV_REQUIRE(f != nullptr, HKV_ERR_ARG, "hkv_fused_forward: null args");
    HKV_REQUIRE(f->num_tokens >= 0, HKV_ERR_ARG, "hkv_fused_forward: num_tokens < 0");
    const int rc = check_fused_source(f, "hkv_fused_forward");
    if (rc != HKV_OK) return rc;
    const HkvPrefillArgs a = fused_as_prefill(f);
    const PfRefSource ref = {f->k_codes, f->v_codes, f->k_scales, f->v_scales, f->k_zps, f->v_zps};
    return prefill_launch(&a, f->num_tokens > 0 ? &ref : nullptr, stream);
}

extern "C" size_t hkv_fused_forward_workspace_bytes(const HkvFusedArgs* f) {
    if (!f || f->num_tokens < 0) return 0;
    const HkvPrefillArgs a = fused_as_prefill(f);
    return hkv_prefill_split_bytes(&a);
}

extern "C" size_t hkv_prefill_split_bytes(const HkvPrefillArgs* a) {
    if (!a || a->batch <= 0 || a->num_kv_heads <= 0 || a->num_q_heads <= 0 || a->num_queries <= 0 ||
        a->num_q_heads % a->num_kv_heads != 0 || a->num_f16_zones < 0 || a->num_f16_zones > HKV_MAX_F16_ZONES)
        return 0;
    const Plan pl = plan_of(a, 1ll << 40);
    if (pl.finish != kFinishPieces) return 0;
    return chunk_ws_bytes(a) + (size_t)pl.state_rows * kStateFloats * sizeof(float);
}

// A state row per (sequence, query head, query), and the causal chunk's K rows and V tiles
// in the zone layout (sized with the query heads, which bound the kv heads).
extern "C" size_t hkv_prefill_workspace_bytes(int32_t batch, int32_t num_q_heads, int32_t num_queries) {
    if (batch <= 0 || num_q_heads <= 0 || num_queries <= 0) return 0;
    const size_t ccap = ((size_t)num_queries + kBlockTokens - 1) / kBlockTokens * kBlockTokens;
    return (size_t)batch * (size_t)num_q_heads * (size_t)num_queries * kStateFloats * sizeof(float) +
           2 * (size_t)batch * (size_t)num_q_heads * ccap * kHeadDim * 2;
}

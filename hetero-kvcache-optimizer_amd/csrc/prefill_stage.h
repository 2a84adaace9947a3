// The staging policies of the chunked-prefill tile loop: fp16 zone and chunk tiles
// (F16Stage), INT4 tiles of the block pool (Int4Stage) and of unpacked codes (RefStage).  Waves 0-3 of a workgroup (team
// 0) stage a tile's K rows, waves 4-7 (team 1) its V^T rows, 16 tokens per wave.
#pragma once

#include "nibble_decode.h"
#include "prefill_flat.h"

#include <math.h>

#include <type_traits>

namespace hkv {

typedef pu4 u4;
typedef pf4 f4;
typedef pu2 u2;

// Staging of INT4 tile x: wave wt of a team handles block wt of the tile (4 blocks of
// 16 tokens), so the block id and record address are wave-uniform (scalar registers,
// one buffer resource per block).  Waves 0-3 lane i: K codes of token i/4, dims
// 32(i%4)..+32, with that row's scale and zero point.  Waves 4-7 lane i: V word
// 4i..4i+3, with the V scales and zero points of tokens 4g..4g+3, g = i/16.
struct SlotK {
    u4 w;
    float ks;
    uint32_t kz;   // zero point in the low byte
};
struct SlotV {
    u4 w;
    f4 vs;
    uint32_t vz;   // zero points of tokens 4g..4g+3 (bytes)
};

// Block id of this wave's block of INT4 tile x (clamped to the last block), the same in
// every lane.  It stays a vector register until it is used two tiles later, so no wait
// for this load sits behind the record loads issued before it.
__device__ __forceinline__ int block_id4(const PrefillParams& p, int nb, int b, int x, int wt) {
    const int lb = min(x * 4 + wt, nb - 1);
    return p.bt[(int64_t)b * p.bt_stride + lb];
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_rsrc(const void* base, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, bytes, 0x00020000);
}
// Buffer resource over this wave's head part of record `id` (an out-of-range id is
// reported and replaced by a valid record).  The range check is a 32-bit unsigned
// compare of a wave-uniform value, and the id used is read back from lane 0, so it and
// the resource stay in scalar registers (a resource the compiler takes for divergent
// wraps every load in a readfirstlane loop).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t part_rsrc(const PrefillParams& p, int h, int id_v) {
    const int id = __builtin_amdgcn_readfirstlane(id_v);
    const bool ok = id >= 0 ? (uint32_t)id < p.pool_blocks : (uint32_t)(~id) < p.staging_blocks;
    const int phys = __builtin_amdgcn_readfirstlane(ok ? id : p.fallback_id);
    if (!ok && p.err && (threadIdx.x & 63) == 0) atomicOr(p.err, 1);
    const int64_t rb = (int64_t)p.Hkv * kHeadPartBytes;
    const uint8_t* part = (phys >= 0 ? p.pool + (int64_t)phys * rb : p.staging + (int64_t)(~phys) * rb) +
                          RecordLayout::part(h);
    return buf_rsrc(part, kHeadPartBytes);
}
__device__ __forceinline__ u4 bld16(__amdgpu_buffer_rsrc_t r, int off) {
    return __builtin_bit_cast(u4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}
__device__ __forceinline__ uint32_t bld4(__amdgpu_buffer_rsrc_t r, int off) {
    return __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0);
}
__device__ __forceinline__ void load_k4(const PrefillParams& p, int h, int id, int lane, SlotK& s) {
    const __amdgpu_buffer_rsrc_t r = part_rsrc(p, h, id);
    const int rr = lane >> 2, pt = lane & 3;
    s.w = bld16(r, kPartKc + rr * 64 + pt * 16);
    s.ks = __uint_as_float(bld4(r, kPartKs + rr * 4));
    s.kz = bld4(r, kPartKz + (rr & ~3)) >> (8 * (rr & 3));   // a word load, no byte value
}
__device__ __forceinline__ void load_v4(const PrefillParams& p, int h, int id, int lane, SlotV& s) {
    const __amdgpu_buffer_rsrc_t r = part_rsrc(p, h, id);
    const int g = lane >> 4;
    s.w = bld16(r, kPartVc + lane * 16);
    s.vs = __builtin_bit_cast(f4, bld16(r, kPartVs + g * 16));
    s.vz = bld4(r, kPartVz + g * 4);
}
// Writes a staged block into LDS: K as (code - zero point) x K scale with the per-token
// biases, V as (code - zero point) x V scale (the queries carry sm_scale x log2 e, so the
// scores come out of the MFMAs in the log2 domain); `valid` = valid tokens of the block.
// Tokens past it get scale 0 (their codes are finite, their scales may be anything) and
// bias -inf.
//
// Rounding.  The products are formed in packed fp16: the scale is rounded to fp16, then
// each product, so a staged element lies within about 1.5 fp16 ulps of the reference's
// dequantized value ((code - zp) x scale in float32, then .to(float16),
// kv_compressor.py:129-132) while the scale is at least 2^-14.  A smaller scale becomes
// an fp16 subnormal with fewer significant bits (about 2% error at 1e-6).  Keeping the
// softmax scale on the queries (not folded into K, which would make every K scale 8x
// smaller) keeps K's scales as far from that range as the reference's own fp16 keys.
__device__ __forceinline__ void store_k4(const SlotK& s, uint8_t* lds, uint8_t* bias, int wt, int lane, int valid) {
    const int rr = lane >> 2, pt = lane & 3;
    const int tok = wt * 16 + rr;
    const uint32_t kz = s.kz & 0xFFu;
    const h2 kz1024 = zp1024(kz, kz), kz64 = zp64(kz, kz);
    const _Float16 f = (_Float16)(rr < valid ? s.ks : 0.0f);
    const h2 f2 = {f, f};
    const uint32_t w4[4] = {s.w.x, s.w.y, s.w.z, s.w.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {          // word j: dims 32pt + 8j .. +8
        const NibPairs a = unpack_word(w4[j], kz1024, kz64);
        *(u4*)(lds + k_addr(tok, pt * 4 + j)) =
            u4{__builtin_bit_cast(uint32_t, a.p0 * f2), __builtin_bit_cast(uint32_t, a.p1 * f2),
               __builtin_bit_cast(uint32_t, a.p2 * f2), __builtin_bit_cast(uint32_t, a.p3 * f2)};
    }
    if (pt == 0) ((float*)bias)[tok] = rr < valid ? 0.0f : -INFINITY;
}
__device__ __forceinline__ void store_v4(const SlotV& s, uint8_t* lds, int wt, int lane, int valid) {
    // V word 4 lane + mm: x0..x3 = tokens 4g..4g+3 at dim c+32mm, x4..x7 at +16
    const int g = lane >> 4, c = lane & 15;
    const h2 z01 = zp1024(s.vz & 0xFFu, (s.vz >> 8) & 0xFFu), z23 = zp64((s.vz >> 16) & 0xFFu, s.vz >> 24);
    const int t0 = 4 * g;
    const h2 vs01 = {(_Float16)(t0 < valid ? s.vs.x : 0.f), (_Float16)(t0 + 1 < valid ? s.vs.y : 0.f)};
    const h2 vs23 = {(_Float16)(t0 + 2 < valid ? s.vs.z : 0.f), (_Float16)(t0 + 3 < valid ? s.vs.w : 0.f)};
    const uint32_t v4[4] = {s.w.x, s.w.y, s.w.z, s.w.w};
    const int unit = wt * 4 + g;
#pragma unroll
    for (int mm = 0; mm < 4; ++mm) {
        const NibPairs a = unpack_word(v4[mm], z01, z23);
        const int d1 = c + 32 * mm, d2 = d1 + 16;
        *(u2*)(lds + vt_addr(d1, unit)) =
            u2{__builtin_bit_cast(uint32_t, a.p0 * vs01), __builtin_bit_cast(uint32_t, a.p1 * vs23)};
        *(u2*)(lds + vt_addr(d2, unit)) =
            u2{__builtin_bit_cast(uint32_t, a.p2 * vs01), __builtin_bit_cast(uint32_t, a.p3 * vs23)};
    }
}

// The INT4 staging policy of the tile loop: two register slots per wave (the records
// of tiles t+2 and t+3 in flight while tile t is attended), block ids fetched one slot
// cycle ahead of their records.
template <int kTeam>
struct Int4Stage {
    static constexpr int kRing = 2;
    typedef typename std::conditional<kTeam == 0, SlotK, SlotV>::type Slot;
    const PrefillParams& p;
    const FlatWave& w;
    const int x0, len;   // the unit's INT4 tiles from x0, tokens up to len
    const int nb4;
    Slot ring[kRing];
    int idn[kRing];   // block id of the tile next loaded into each slot

    __device__ Int4Stage(const PrefillParams& p_, const TileMap& tm, const FlatWave& w_, int x0_, int x1_)
        : p(p_), w(w_), x0(x0_), len(min(tm.len4, x1_ * kPfT)), nb4((len + kBlockTokens - 1) / kBlockTokens) {}
    // valid tokens of this wave's block of tile x and of tile x, branch-free (0 past the end)
    __device__ int valid(int x) const { return min(kBlockTokens, max(0, len - ((x0 + x) * 4 + w.wt) * kBlockTokens)); }
    __device__ int tvalid(int x) const { return min(kPfT, max(0, len - (x0 + x) * kPfT)); }
    __device__ void load(int id, Slot& sl) const {
        if constexpr (kTeam == 0) load_k4(p, w.h, id, w.lane, sl);
        else load_v4(p, w.h, id, w.lane, sl);
    }
    __device__ void stage(int s, uint8_t* buf, uint8_t* bias, int x) const {
        if constexpr (kTeam == 0) store_k4(ring[s], buf, bias, w.wt, w.lane, valid(x));
        else store_v4(ring[s], buf, w.wt, w.lane, valid(x));
    }
    __device__ void refill(const TileMap&, int s, int x) {   // tile x just staged from slot s
        load(idn[s], ring[s]);
        idn[s] = block_id4(p, nb4, w.b, x0 + x + 2 * kRing, w.wt);
    }
    __device__ void start(const TileMap& tm, uint8_t* lds) {
#pragma unroll
        for (int x = 0; x < kRing; ++x) {
            load(block_id4(p, nb4, w.b, x0 + x, w.wt), ring[x]);
            idn[x] = block_id4(p, nb4, w.b, x0 + x + kRing, w.wt);
        }
#pragma unroll
        for (int x = 0; x < kRing; ++x) {
            stage(x, flat_buf(lds, x), flat_bias(lds, x), x);
            refill(tm, x, x);
        }
    }
    __device__ void mask(int, pf16v (&)[2]) const {}
    __device__ const uint8_t* values(int, const uint8_t* buf, uint8_t*) const { return buf; }
};

// The fp16 staging policy of the tile loop: one register slot per wave (64 bytes per
// lane: a quarter of a tile's K rows or of its V tiles).  A cursor walks the sources one
// tile per load, so that a tile costs one scalar compare in the common case (finding the
// source of each tile from the tile counts, three times per tile, was ~100 scalar
// instructions and branches); the loads go through buffer resources that end with the
// tile's valid tokens, so rows past them read as zeros.
template <int kTeam>
struct F16Stage {
    static constexpr int kRing = 1;
    const PrefillParams& p;
    const FlatWave& w;
    const int chunk0;      // the loop's tile of the chunk's first tokens (past every tile without a chunk)
    const int last;        // the last tile that a query of the wave sees (past every tile without a chunk)
    int tiles;             // tiles not yet loaded
    int si, left, len;     // the source, its tiles not yet loaded, its tokens from the next tile on
    const uint16_t* base;  // the next tile's K rows (team 0) or V tiles (team 1)
    int q0, q1, q2;        // valid tokens of the tile attended, the one staged after it, the slot's
    u4 slot[4];

    __device__ F16Stage(const PrefillParams& p_, const TileMap& tm, const FlatWave& w_, int x0, int x1)
        : p(p_), w(w_), chunk0(tm.nc > 0 ? tm.nz_t[0] + tm.nz_t[1] + tm.nz_t[2] - x0 : 1 << 24),
          last(chunk0 + w_.q_hi / kPfT), tiles(x1 - x0) {
        si = 0;
        int x = x0;
#pragma unroll
        for (int zi = 0; zi < HKV_MAX_F16_ZONES; ++zi)
            if (si == zi && x >= tm.nz_t[zi]) {   // zones without a tile are passed over
                x -= tm.nz_t[zi];
                si = zi + 1;
            }
        open(tm, x);
    }
    __device__ int len_of(const TileMap& tm, int i) const {
        return i == 0 ? tm.lenz[0] : i == 1 ? tm.lenz[1] : i == 2 ? tm.lenz[2] : p.Sq;
    }
    // The cursor at tile xl of source si.
    __device__ void open(const TileMap& tm, int xl) {
        const PfSrc& s = p.src[si];
        const int64_t row = ((int64_t)w.b * p.Hkv + w.h) * s.cap + (int64_t)xl * kPfT;   // capacities are multiples of 16
        base = (kTeam == 0 ? s.k : s.v) + row * kHeadDim;
        len = len_of(tm, si) - xl * kPfT;
        left = (len + kPfT - 1) / kPfT;
    }
    // Loads the next tile (none: an empty one) and returns its valid tokens.
    __device__ int load_into(const TileMap& tm, u4 (&dst)[4]) {
        if (left == 0 && tiles > 0) {
            do ++si;
            while (si < HKV_MAX_F16_ZONES && len_of(tm, si) == 0);
            open(tm, 0);
        }
        const int nv = tiles > 0 ? min(len, kPfT) : 0;
        // K: wave wt's 16 rows (256 bytes each), lane i row i / 4, dims 32 (i % 4) .. +32.  V: its
        // 16-token tile (4 KB), lane i bytes 64 i: halves [n][i] = V[4g + i][c + 16n]
        const int bytes = kTeam == 0 ? nv * (kHeadDim * 2)
                                     : (nv + kBlockTokens - 1) / kBlockTokens * (kBlockTokens * kHeadDim * 2);
        const __amdgpu_buffer_rsrc_t r = buf_rsrc(base, bytes);
        const int off = w.wt * (kBlockTokens * kHeadDim * 2) + w.lane * 64;
#pragma unroll
        for (int j = 0; j < 4; ++j) dst[j] = bld16(r, off + 16 * j);
        base += kPfT * kHeadDim;
        len -= kPfT;
        --left;
        --tiles;
        return nv;
    }
    __device__ int tvalid(int) const { return q0; }
    __device__ void put(const u4 (&d)[4], uint8_t* buf, uint8_t* bias, int nv) const {
        if constexpr (kTeam == 0) {
            const int tok = w.wt * 16 + (w.lane >> 2), pt = w.lane & 3;
#pragma unroll
            for (int j = 0; j < 4; ++j) *(u4*)(buf + k_addr(tok, pt * 4 + j)) = d[j];
            if (pt == 0) ((float*)bias)[tok] = tok < nv ? 0.0f : -INFINITY;
        } else {
            // V^T rows c + 16n, unit 4 wt + g (tokens 16 wt + 4g .. +3); tokens past the
            // length are cleared so masked probabilities multiply finite values
            const int g = w.lane >> 4, c = w.lane & 15;
            const int t0 = w.wt * 16 + 4 * g;
            const uint32_t m01 = (t0 + 0 < nv ? 0x0000FFFFu : 0u) | (t0 + 1 < nv ? 0xFFFF0000u : 0u);
            const uint32_t m23 = (t0 + 2 < nv ? 0x0000FFFFu : 0u) | (t0 + 3 < nv ? 0xFFFF0000u : 0u);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                *(u2*)(buf + vt_addr(c + 32 * j, w.wt * 4 + g)) = u2{d[j].x & m01, d[j].y & m23};
                *(u2*)(buf + vt_addr(c + 32 * j + 16, w.wt * 4 + g)) = u2{d[j].z & m01, d[j].w & m23};
            }
        }
    }
    __device__ void stage(int, uint8_t* buf, uint8_t* bias, int) const { put(slot, buf, bias, q2); }
    __device__ void refill(const TileMap& tm, int, int) {
        q0 = q1;
        q1 = q2;
        q2 = load_into(tm, slot);
    }
    __device__ void start(const TileMap& tm, uint8_t* lds) {
        // tiles 0 and 1 requested together: one load round trip before the loop, not two
        u4 next[4];
        q0 = load_into(tm, slot);
        q1 = load_into(tm, next);
        put(slot, flat_buf(lds, 0), flat_bias(lds, 0), q0);
        q2 = load_into(tm, slot);
        put(next, flat_buf(lds, 1), flat_bias(lds, 1), q1);
    }
    // Chunk tile xl: token t (chunk position xl * 64 + t) is visible to query qrow when
    // xl * 64 + t <= qrow; a wave whose lowest query is past the tile needs no mask.
    __device__ void mask(int x, pf16v (&S)[2]) const {
        if ((x - chunk0) * kPfT + (kPfT - 1) > w.q_lo) {
            const int lim = w.qrow - (x - chunk0) * kPfT;
#pragma unroll
            for (int tb = 0; tb < 2; ++tb)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    if (tb * 32 + 8 * (r >> 2) + 4 * w.hh + (r & 3) > lim) S[tb][r] = -INFINITY;
        }
    }
    // Past the wave's last query the probabilities are zeros, but the loop's rounds go on for up
    // to three tiles: a non-finite value of a token there would turn the wave's outputs to NaN
    // (0 x inf), so these tiles weigh zeros.  Within the last tile it does, as in any product
    // with masked probabilities.
    __device__ const uint8_t* values(int x, const uint8_t* buf, uint8_t* lds) const {
        return x > last ? lds + kFlatLdsBytes - kVOff : buf;
    }
};

// The staging policy of unpacked INT4 codes: the same staged values as Int4Stage, from one
// byte per code.  Reading the codes directly, twice the packed bytes, costs less than
// clearing a pool, repacking the codes into it and reading that (512 queries of 32/32 heads
// over 4096 keys: 90 -> 64 us a call).  A tile takes ~7% longer than a packed one: twice the
// code words to load and unpack.  kVec: rows of a multiple of 4 tokens, whose scales and zero
// points load as vectors, which leaves registers for a second tile in flight.
template <int kTeam, bool kVec>
struct RefStage {
    static constexpr int kRing = kVec ? 2 : 1;
    const PrefillParams& p;
    const FlatWave& w;
    const int x0, len;     // the unit's tiles from x0, tokens up to len
    struct Slot {
        u4 a, b;           // team 0: this lane's 32 K codes; team 1: 4 tokens x (4 + 4) V codes
        f4 sc;             // scales (team 0: one)
        uint32_t zp;       // zero points, one per byte
    } ring[kRing];

    __device__ RefStage(const PrefillParams& p_, const TileMap& tm, const FlatWave& w_, int x0_, int x1_)
        : p(p_), w(w_), x0(x0_), len(min(tm.len4, x1_ * kPfT)) {}
    __device__ int tvalid(int x) const { return min(kPfT, max(0, len - (x0 + x) * kPfT)); }
    // Requests tile x.  The resources end with its valid rows: what lies past them reads as
    // zero (scale 0: staged as zeros).
    __device__ void load(int x, Slot& s) const {
        const int nv = tvalid(x);
        const int64_t row = ((int64_t)w.b * p.Hkv + w.h) * p.int4_max_len + (int64_t)(x0 + x) * kPfT;
        const uint8_t *codes = kTeam == 0 ? p.ref.kc : p.ref.vc, *zps = kTeam == 0 ? p.ref.kz : p.ref.vz;
        const float* scales = kTeam == 0 ? p.ref.ks : p.ref.vs;
        const __amdgpu_buffer_rsrc_t rc = buf_rsrc(codes + row * kHeadDim, nv * kHeadDim);
        const __amdgpu_buffer_rsrc_t rs = buf_rsrc(scales + row, nv * 4), rz = buf_rsrc(zps + row, nv);
        if constexpr (kTeam == 0) {
            // token 16 wt + lane / 4, dims 32 (lane % 4) .. +32
            const int tok = w.wt * 16 + (w.lane >> 2), off = tok * kHeadDim + (w.lane & 3) * 32;
            s.a = bld16(rc, off);
            s.b = bld16(rc, off + 16);
            s.sc[0] = __uint_as_float(bld4(rs, tok * 4));
            s.zp = __builtin_amdgcn_raw_buffer_load_b8(rz, tok, 0, 0);
        } else {
            // tokens 16 wt + 4g .. +3, dims 4c .. +3 and 64 + 4c .. +3 (g = lane / 16, c = lane % 16)
            const int t0 = w.wt * 16 + (w.lane >> 4) * 4, off = t0 * kHeadDim + (w.lane & 15) * 4;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                s.a[t] = bld4(rc, off + t * kHeadDim);
                s.b[t] = bld4(rc, off + t * kHeadDim + 64);
            }
            if constexpr (kVec) {
                s.sc = __builtin_bit_cast(f4, bld16(rs, t0 * 4));
                s.zp = bld4(rz, t0);
            } else {
                s.zp = 0u;
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    s.sc[t] = __uint_as_float(bld4(rs, (t0 + t) * 4));
                    s.zp |= (uint32_t)__builtin_amdgcn_raw_buffer_load_b8(rz, t0 + t, 0, 0) << (8 * t);
                }
            }
        }
    }
    // (code - zero point) x scale as Int4Stage stages it: the scale rounded to fp16, then the
    // product.  Only the low four bits of a code count, as in the packed pool.
    __device__ void stage(int slot, uint8_t* buf, uint8_t* bias, int x) const {
        const Slot& s = ring[slot];
        if constexpr (kTeam == 0) {
            const int tok = w.wt * 16 + (w.lane >> 2), pt = w.lane & 3;
            const _Float16 f = (_Float16)s.sc[0];
            const fh2 f2 = {f, f}, z = zp1024(s.zp, s.zp);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                u4 o;
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const uint32_t m = (j < 2 ? s.a : s.b)[2 * (j & 1) + e] & 0x0F0F0F0Fu;
                    const fh2 lo = __builtin_bit_cast(fh2, __builtin_amdgcn_perm(0x64646464u, m, 0x04010400u)) - z;
                    const fh2 hi = __builtin_bit_cast(fh2, __builtin_amdgcn_perm(0x64646464u, m, 0x04030402u)) - z;
                    o[2 * e] = __builtin_bit_cast(uint32_t, lo * f2);
                    o[2 * e + 1] = __builtin_bit_cast(uint32_t, hi * f2);
                }
                *(u4*)(buf + k_addr(tok, pt * 4 + j)) = o;
            }
            if (pt == 0) ((float*)bias)[tok] = tok < tvalid(x) ? 0.0f : -INFINITY;
        } else {
            // lane c's four dims of a word are written starting at the (c / 4)-th: 16 lanes then
            // write 16 rows on banks of their own (all starting at the first: 4 rows per bank,
            // 2.25 against 2.0 us per tile)
            const int unit = w.wt * 4 + (w.lane >> 4), c = w.lane & 15, r = c >> 2;
            const fh2 z01 = zp1024(s.zp & 0xffu, (s.zp >> 8) & 0xffu), z23 = zp1024((s.zp >> 16) & 0xffu, s.zp >> 24);
            const fh2 f01 = {(_Float16)s.sc[0], (_Float16)s.sc[1]}, f23 = {(_Float16)s.sc[2], (_Float16)s.sc[3]};
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                u4 v = e < 4 ? s.a : s.b;
#pragma unroll
                for (int t = 0; t < 4; ++t) v[t] = __builtin_amdgcn_alignbyte(v[t], v[t], r);
                const uint32_t sel = 0x0C000C00u | (uint32_t)(e & 3) | ((uint32_t)(4 + (e & 3)) << 16);
                const uint32_t m01 = and_or(__builtin_amdgcn_perm(v[1], v[0], sel), 0x000F000Fu, 0x64006400u);
                const uint32_t m23 = and_or(__builtin_amdgcn_perm(v[3], v[2], sel), 0x000F000Fu, 0x64006400u);
                *(u2*)(buf + vt_addr((e < 4 ? 0 : 64) + 4 * c + ((e + r) & 3), unit)) =
                    u2{__builtin_bit_cast(uint32_t, (__builtin_bit_cast(fh2, m01) - z01) * f01),
                       __builtin_bit_cast(uint32_t, (__builtin_bit_cast(fh2, m23) - z23) * f23)};
            }
        }
    }
    __device__ void refill(const TileMap&, int slot, int x) { load(x + kRing, ring[slot]); }
    __device__ void start(const TileMap&, uint8_t* lds) {
#pragma unroll
        for (int x = 0; x < kRing; ++x) load(x, ring[x]);
#pragma unroll
        for (int x = 0; x < 2; ++x) {
            stage(x % kRing, flat_buf(lds, x), flat_bias(lds, x), x);
            load(x + kRing, ring[x % kRing]);
        }
    }
    __device__ void mask(int, pf16v (&)[2]) const {}
    __device__ const uint8_t* values(int, const uint8_t* buf, uint8_t*) const { return buf; }
};

}  // namespace hkv

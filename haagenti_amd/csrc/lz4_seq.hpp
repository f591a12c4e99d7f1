// Raw-LZ4 block decoding, one wavefront per block, in batches of sequences:
// a scalar pass parses up to 64 sequences into lane-held descriptors, a wave
// prefix sum turns their lengths into output offsets, and the copies of the
// whole batch then run lane-parallel -- every literal run of the batch in one
// set of passes, then the matches, those that read only bytes final before
// them sharing a pass.  Used by the batched LZ4 kernel (lz4_seq.hip) and the
// fused LZ4 -> tile kernel (hctt_decode.hip).
//
// What bounds it: one block is one wave's chain of dependent instructions
// (7-10 cycles each when the wave is alone on its SIMD).  Tiles of 10 %
// retention make ~1,400 sequences of ~10 bytes a 16 KiB block; a tensor of
// 652 such blocks took 607 us when every sequence's header was read on its
// own and matches were copied in runs up to the first that reads one of
// them, 174 us with the tokens found by a walk (about 110 cycles a sequence),
// one lane copying a sequence's literals and its match, and matches going as
// soon as their own source bytes are there: 3.5 rounds a batch of 64.  At
// 15 % 268 -> 128 us, at 20 % 102 -> 88 us, at 24 % (16 long sequences a
// block) 59 -> 53.
//
// Semantics: crates/haagenti-lz4/src/block.rs:261-366 (decompress_block):
// the same checks in the same order, the same reported positions, the early
// stop once the output reaches output_size.  Every check is made by the
// parse, so a batch's copies never fail; a block that fails is not copied
// further (its caller zero-fills its output).
//
// LDS per wave:
//  * an output ring of R bytes holding the block's latest output.  A match
//    reads its source from the ring when the source was written at most
//    R - 32 bytes before the end of the current batch (nothing of the batch
//    has overwritten it), else from the output in global memory, which every
//    complete 16-byte chunk has reached by then (batches produce at most
//    R - 64 bytes and complete chunks are written out after each batch);
//  * an input stage of S bytes of the compressed stream, refilled with
//    16-byte loads; headers and literal runs are read there.  A batch ends
//    where the stage does; a literal run or match that crosses a batch end
//    continues in the next batch;
//  * a table that maps a pass's chunks to their runs, or marks the output
//    bytes of the matches still to be copied.
// Copies write exactly their own bytes (16-byte chunks aligned in output
// position; partial dwords merged with LDS and/or atomics), so the runs of a
// pass may share chunks.  A match of length n at output position v with
// offset `off` writes byte t from position v - off + (t mod off): a periodic
// (overlapping) match reads only the `off` bytes before it, so all of its
// chunks are independent.  Matches of one pass read only bytes before the
// first of them.
//
// With LDS = true the whole block output stays in the ring (a block of at
// most R - 32 bytes; every match reads the ring, nothing is written out) for
// a consumer that reads it there; progress(op) runs after each batch with
// the output before op final.
#pragma once

#include "hh_internal.hpp"

namespace hh {
namespace seq {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
// LDS-qualified pointers: every ring, stage and table access is a ds_*
// instruction (a generic pointer lets the compiler merge a ring read with a
// global read into one flat load, which is not ordered after earlier ds_*
// writes of other lanes)
typedef __attribute__((address_space(3))) uint8_t lds8;
typedef __attribute__((address_space(3))) uint32_t lds32;
typedef __attribute__((address_space(3))) u32x4 ldsx4;

__device__ __forceinline__ uint32_t rfl(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ uint32_t rdl(uint32_t v, uint32_t l) { return __builtin_amdgcn_readlane(v, l); }
__device__ __forceinline__ uint64_t ballot(bool b) { return __builtin_amdgcn_ballot_w64(b); }
__device__ __forceinline__ uint32_t bperm(uint32_t v, uint32_t l) {
    return (uint32_t)__builtin_amdgcn_ds_bpermute((int)(l << 2), (int)v);
}

// Inclusive prefix sum / maximum over the 64 lanes: DPP row shifts (1, 2,
// 4, 8 within each row of 16 lanes) and the row broadcasts of lanes 15 and
// 31; lanes whose source lies outside the row keep the 0 passed as `old`.
__device__ __forceinline__ uint32_t scan_add(uint32_t v) {
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false);
    return v;
}
__device__ __forceinline__ uint32_t scan_max(uint32_t v) {
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false));
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false));
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false));
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false));
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false));
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false));
    return v;
}

// Orders the LDS accesses of the wave's lanes: what one lane wrote before it
// is what every lane reads after it (the compiler may otherwise keep a
// value a lane stored itself and miss another lane's atomic update).
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// 16 bytes starting at byte sh of the 20 bytes d0..d4.
__device__ __forceinline__ u32x4 realign(const uint32_t (&d)[5], uint32_t sh) {
    return u32x4{__builtin_amdgcn_alignbyte(d[1], d[0], sh), __builtin_amdgcn_alignbyte(d[2], d[1], sh),
                 __builtin_amdgcn_alignbyte(d[3], d[2], sh), __builtin_amdgcn_alignbyte(d[4], d[3], sh)};
}

// Byte mask of bytes [lo, hi) of dword i of a 16-byte chunk.
__device__ __forceinline__ uint32_t dword_mask(uint32_t lo, uint32_t hi, uint32_t i) {
    const int32_t a = (int32_t)lo - (int32_t)(4 * i), b = (int32_t)hi - (int32_t)(4 * i);
    const uint32_t ma = a <= 0 ? 0xffffffffu : a >= 4 ? 0u : (0xffffffffu << (8 * a));
    const uint32_t mb = b >= 4 ? 0xffffffffu : b <= 0 ? 0u : ((1u << (8 * b)) - 1u);
    return ma & mb;
}

// x mod m for 0 <= x < 2^24, 1 <= m < 2^17 (f32 quotient estimate, corrected).
__device__ __forceinline__ uint32_t umod(uint32_t x, uint32_t m) {
    uint32_t q = (uint32_t)((float)x * __builtin_amdgcn_rcpf((float)m));
    int32_t r = (int32_t)(x - q * m);
    r = r < 0 ? r + (int32_t)m : r;
    r = r >= (int32_t)m ? r - (int32_t)m : r;
    r = r < 0 ? r + (int32_t)m : r;
    return (uint32_t)r;
}

// Parse state between batches.
enum : uint32_t { kToken = 0, kLitExt = 1, kLit = 2, kOff = 3, kMatchExt = 4, kMatch = 5 };

struct NoProgress {
    __device__ __forceinline__ void operator()(uint32_t) const {}
};

template <uint32_t R, uint32_t S, bool LDS>
struct SeqDec {
    static_assert((R & (R - 1)) == 0 && R >= 4096, "ring size is a power of two");
    static_assert(S % 1024 == 0 && S >= 1024, "stage is whole KiB");
    static constexpr uint32_t kRM = R - 1;
    static constexpr uint32_t kS = S;
    static constexpr uint32_t kOB = LDS ? R - 32 : R - 96;  // batch output budget
    static constexpr uint32_t kSFront = 16;                // stage under-read (first chunk of a literal)
    static constexpr uint32_t kSPad = 32;                  // stage over-read (headers, realign)
    static constexpr uint32_t kStageLds = kSFront + S + kSPad;
    // (with a stage of 8 KiB the table fills a wave's area of the fused
    // kernel, 12 of which leave room for 3 block buffers)
    static constexpr uint32_t kTabWords = 112;
    static constexpr uint32_t kTabLds = 4 * kTabWords;
    static constexpr uint32_t kList = 256;
    // batches whose matches may run in any order (match_short): their output
    // bytes each have a bit in the table, and one word after them
    static constexpr uint32_t kShortBytes = 32 * (kTabWords - 1);
    static constexpr uint32_t kShortLit = 32;    // longest literal run copied by one lane
    static constexpr uint32_t kShortMatch = 18;  // longest match without a length extension
    // ring, table, stage (the caller may place them elsewhere)
    static constexpr uint32_t kLds = R + kTabLds + kStageLds;

    lds8 *ring;
    lds32 *tab;           // kTabWords words
    uint32_t list;        // up to kList distances from a token to the next: entry i in byte i / 64 of lane i % 64
    lds8 *stage;          // kSFront bytes of slack before it, kSPad after
    const uint8_t *gbuf;  // whole input buffer: every read is clamped to it
    uint64_t gsz;
    uint64_t ioff;        // block start in gbuf
    uint8_t *obase;       // 16-aligned, <= the block's output address
    uint32_t a0;          // output address - obase
    uint32_t cap;
    // Block-relative input position of stage byte 0, modulo 2^32 (up to 15
    // before the block start when the block starts unaligned).
    uint32_t sb;
    bool at_end;          // the stage reaches the end of the input buffer
    uint32_t op;          // bytes decoded
    uint32_t fl;          // bytes written out
    int lane;

    // ---------------------------------------------------------------- stage
    // The stage holds input bytes [sb, sb + S) (block-relative; sb is
    // 16-aligned in memory, up to 15 bytes before the block when it starts
    // unaligned).  The next stage, starting 64 bytes before this one ends,
    // is loaded into registers (pv) as soon as this one is in place, so its
    // loads are in flight while the wave parses and copies.
    u32x4 pv[S / 1024];
    uint32_t pf;   // input position of the prefetched stage
    bool pf_on;    // pv holds (or is loading) the stage at pf
    // Loads into v the stage whose byte 0 is input byte s0 (16-aligned in
    // memory).  Inside the buffer: 16-byte loads; at its edges each dword is
    // read at an address clamped to the dwords holding buffer bytes (bytes
    // outside the buffer are never used).
    __device__ __forceinline__ void load_stage(uint32_t s0, u32x4 (&v)[S / 1024]) const {
        const int64_t b0 = (int64_t)ioff + (int64_t)(int32_t)s0;
        if (b0 >= 0 && b0 + (int64_t)S <= (int64_t)gsz) {
#pragma unroll
            for (uint32_t i = 0; i < S / 1024; i++)
                v[i] = *reinterpret_cast<const u32x4 *>(gbuf + b0 + 16 * (lane + 64 * i));
        } else {
            const int64_t lo = -(int64_t)((uintptr_t)gbuf & 3u);
            const int64_t hi = (int64_t)(((uintptr_t)gbuf + gsz - 1) & ~(uintptr_t)3) - (int64_t)(uintptr_t)gbuf;
#pragma unroll
            for (uint32_t i = 0; i < S / 1024; i++) {
#pragma unroll
                for (uint32_t j = 0; j < 4; j++) {
                    int64_t o = b0 + 16 * (lane + 64 * i) + 4 * j;
                    o = o < lo ? lo : o > hi ? hi : o;
                    v[i][j] = *reinterpret_cast<const uint32_t *>(gbuf + o);
                }
            }
        }
    }
    __device__ __forceinline__ void put_stage(uint32_t s0, const u32x4 (&v)[S / 1024]) {
        sb = s0;
        at_end = (int64_t)ioff + (int64_t)(int32_t)s0 + (int64_t)S >= (int64_t)gsz;
#pragma unroll
        for (uint32_t i = 0; i < S / 1024; i++)
            *reinterpret_cast<ldsx4 *>(stage + 16 * (lane + 64 * i)) = v[i];
        wave_sync();
    }
    // Starts the load of the stage after the current one.  Not in LDS mode,
    // whose caller runs other waves beside this one to hide the loads (and
    // needs the registers).
    static constexpr bool kPrefetch = !LDS;
    __device__ __forceinline__ void prefetch() {
        pf_on = kPrefetch && !at_end;
        if (pf_on) {
            pf = sb + S - 64u;
            load_stage(pf, pv);
        }
    }
    // Makes the stage hold input position x: from the prefetched stage when
    // it holds x with at least 1 KiB after it, else loaded now.
    __device__ __forceinline__ void restage(uint32_t x) {
        if constexpr (kPrefetch) {
            if (!(pf_on && x - pf <= S - 1024u)) {
                pf = x - (uint32_t)((uintptr_t)(gbuf + ioff + x) & 15u);
                load_stage(pf, pv);
            }
            put_stage(pf, pv);
            prefetch();
        } else {
            const uint32_t s0 = x - (uint32_t)((uintptr_t)(gbuf + ioff + x) & 15u);
            u32x4 v[S / 1024];
            load_stage(s0, v);
            put_stage(s0, v);
        }
    }
    // [x, x + 8) is in the stage (or the stage reaches the end of the buffer)
    __device__ __forceinline__ bool in_stage8(uint32_t x) const { return at_end || x - sb <= S - 8; }
    // stage bytes available for a literal run from x on
    __device__ __forceinline__ uint32_t lit_avail(uint32_t x) const { return at_end ? 0xffffffffu : sb + S - x; }

    // Header window: input bytes [hb, hb + hv) in scalar registers (hv <=
    // 16), read from the stage 16 at a time, so that a sequence's offset,
    // its match-length bytes and the next token usually come from one read.
    uint64_t hw0, hw1;
    uint32_t hb, hv;
    // 16 bytes from x on (x in the stage); the bytes past the stage's data
    // are not counted valid
    __device__ __forceinline__ void read16(uint32_t x) {
        const uint32_t so = x - sb;
        const lds32 *q = reinterpret_cast<const lds32 *>(stage + (so & ~3u));
        const uint32_t d0 = q[0], d1 = q[1], d2 = q[2], d3 = q[3], d4 = q[4];
        const uint32_t sh = so & 3u;
        const uint32_t w0 = rfl(__builtin_amdgcn_alignbyte(d1, d0, sh));
        const uint32_t w1 = rfl(__builtin_amdgcn_alignbyte(d2, d1, sh));
        const uint32_t w2 = rfl(__builtin_amdgcn_alignbyte(d3, d2, sh));
        const uint32_t w3 = rfl(__builtin_amdgcn_alignbyte(d4, d3, sh));
        hw0 = ((uint64_t)w1 << 32) | w0;
        hw1 = ((uint64_t)w3 << 32) | w2;
        hb = x;
        hv = at_end || S - so >= 16u ? 16u : S - so;
    }
    // 8 bytes from x on: from the window when it holds them, else from the
    // stage (the caller has checked in_stage8(x)).
    __device__ __forceinline__ bool in_win8(uint32_t x) const { return x - hb <= hv - 8u && hv >= 8u; }
    __device__ __forceinline__ uint64_t peek8(uint32_t x) const {  // in_win8(x)
        const uint32_t k = x - hb;  // 0..8
        const uint64_t a = hw0 >> (8 * (k & 7u)), b = (hw1 << 1) << (63 - 8 * (k & 7u));
        return k >= 8u ? hw1 : (a | b);
    }
    __device__ __forceinline__ uint64_t get8(uint32_t x) {
        if (!in_win8(x)) read16(x);
        return peek8(x);
    }
    // the raw stage read of 8 bytes (extension runs)
    __device__ __forceinline__ uint64_t read8(uint32_t x) {
        read16(x);
        return hw0;
    }

    // Length extension from *pp (block.rs:277-289, 329-341) once 7 (or 6)
    // 0xFF bytes have been seen: adds 255 per 0xFF byte plus the first other
    // byte.  Returns 0 when done, 1 at the end of the block input (the
    // reference reports UnexpectedEof), 2 where it goes on past the stage
    // (the caller restages there or, where the batch holds copies that read
    // the stage, ends the batch and parses the sequence again).
    __device__ __forceinline__ int ext_slow(uint32_t &pp, uint32_t end, uint64_t &len) {
        uint32_t p = pp;
        for (;;) {
            pp = p;
            if (p >= end) return 1;
            if (!in_stage8(p)) return 2;
            const uint64_t x = read8(p);
            const uint64_t nz = ~x;
            if (nz == 0) {
                len += 255ull * 8;
                p += 8;
                continue;
            }
            const uint32_t e = (uint32_t)__builtin_ctzll(nz) >> 3;
            if (p + e >= end) return 1;
            len += 255ull * e + ((x >> (8 * e)) & 0xffu);
            pp = p + e + 1;
            return 0;
        }
    }

    // ---------------------------------------------------------------- copies
    // Writes bytes [lo, hi) of chunk o to the ring at virtual position cv
    // (16-aligned); bytes outside [lo, hi) are left as they are (a chunk's
    // partial dwords are merged with LDS and / or atomics, so two lanes may
    // share a chunk).
    __device__ __forceinline__ void mwrite(uint32_t cv, const u32x4 &o, uint32_t lo, uint32_t hi) {
        lds8 *dst = ring + (cv & kRM);
        if (lo == 0 && hi == 16) {
            *reinterpret_cast<ldsx4 *>(dst) = o;
        } else {
#pragma unroll
            for (uint32_t i = 0; i < 4; i++) {
                const uint32_t m = dword_mask(lo, hi, i);
                lds32 *w = reinterpret_cast<lds32 *>(dst + 4 * i);
                __hip_atomic_fetch_and(w, ~m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                __hip_atomic_fetch_or(w, o[i] & m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            }
        }
    }

    // 16 bytes of output from virtual position sp on: from the ring when
    // their 20-byte window (from sp rounded down to 4) starts at or after
    // rlo (written less than R bytes before the batch end, see execute), else
    // from the written-out output.  The output's dwords are read at addresses clamped
    // to the dwords holding the block's output bytes, so a window reaching
    // outside them reads no memory outside them (those bytes are never used:
    // they lie before a match's source).
    __device__ __forceinline__ u32x4 src16(int32_t sp, int32_t rlo) const {
        const int32_t w = sp & ~3;
        uint32_t d[5];
        if (LDS || w >= rlo) {
#pragma unroll
            for (int i = 0; i < 5; i++) d[i] = *reinterpret_cast<const lds32 *>(ring + (((uint32_t)w + 4u * i) & kRM));
        } else {
            const int32_t lo = (int32_t)(a0 & ~3u), hi = (int32_t)((a0 + cap - 1u) & ~3u);
#pragma unroll
            for (int i = 0; i < 5; i++) {
                int32_t x = w + 4 * i;
                x = x < lo ? lo : x > hi ? hi : x;
                d[i] = *reinterpret_cast<const uint32_t *>(obase + x);
            }
        }
        return realign(d, (uint32_t)sp & 3u);
    }

    // Chunk c of the literal run of n bytes at virtual position v whose
    // bytes are at stage offset src.
    __device__ __forceinline__ void lit_chunk(uint32_t v, uint32_t n, uint32_t src, uint32_t c) {
        const uint32_t cv = (v & ~15u) + 16u * c;
        const uint32_t lo = v > cv ? v - cv : 0u;
        const uint32_t hi = v + n - cv < 16u ? v + n - cv : 16u;
        const int32_t sp = (int32_t)(src + cv - v);  // >= src - 15
        const lds32 *q = reinterpret_cast<const lds32 *>(stage + (sp & ~3));
        uint32_t d[5];
#pragma unroll
        for (int i = 0; i < 5; i++) d[i] = q[i];
        mwrite(cv, realign(d, (uint32_t)sp & 3u), lo, hi);
    }

    // Chunk c of the match of n bytes at virtual position v, offset off.
    // Byte t of the match comes from v - off + (t mod off).  K: 0 a plain
    // copy (off >= n), 1 periodic with off >= 16, 2 periodic with off < 16,
    // -1 chosen per chunk (the runs of a pass differ).
    template <int K>
    __device__ __forceinline__ void match_chunk(uint32_t v, uint32_t n, uint32_t off, uint32_t c, int32_t rlo) {
        const uint32_t cv = (v & ~15u) + 16u * c;
        const uint32_t lo = v > cv ? v - cv : 0u;
        const uint32_t hi = v + n - cv < 16u ? v + n - cv : 16u;
        const int32_t r0 = (int32_t)(cv - v);  // match-relative position of chunk byte 0, >= -15
        u32x4 o;
        const int k = K >= 0 ? K : (r0 + (int32_t)hi <= (int32_t)off ? 0 : off >= 16u ? 1 : 2);
        if (k == 0) {
            // every byte of the chunk lies in the first period
            o = src16((int32_t)(cv - off), rlo);
        } else if (k == 1) {
            // byte t from v - off + ((a + t) mod off), wrapping at most once:
            // bytes before the wrap from base on, the rest from base - off on
            const uint32_t a = umod((uint32_t)(r0 + (int32_t)off), off);
            const int32_t base = (int32_t)(v - off + a);
            o = src16(base, rlo);
            const u32x4 b = src16(base - (int32_t)off, rlo);
            const uint32_t kw = off - a < 16u ? off - a : 16u;  // bytes before the wrap
#pragma unroll
            for (uint32_t i = 0; i < 4; i++) {
                const uint32_t m = dword_mask(0, kw, i);
                o[i] = (o[i] & m) | (b[i] & ~m);
            }
        } else {
            // byte t from v - off + ((a + t) mod off), in the ring
            uint32_t m = umod((uint32_t)(r0 + 16 * (int32_t)off), off);
            const uint32_t sv = v - off;
            uint32_t d[4] = {0u, 0u, 0u, 0u};
#pragma unroll
            for (uint32_t t = 0; t < 16; t++) {
                d[t >> 2] |= (uint32_t)ring[(sv + m) & kRM] << (8 * (t & 3));
                m = m + 1 == off ? 0u : m + 1;
            }
            o = u32x4{d[0], d[1], d[2], d[3]};
        }
        mwrite(cv, o, lo, hi);
    }

    // Lane l's run for flat chunk g0 + l, given each run's first flat chunk
    // `ex` (runs in lane order, ex non-decreasing): the last run i with
    // ex_i <= g0 + l.  Runs starting in [g0, g0 + 64) mark their first lane
    // in the table (largest index wins), a prefix maximum spreads them, and
    // the runs started before g0 (a prefix of the lanes) set the floor.
    __device__ __forceinline__ uint32_t lane_run(uint32_t ex, uint32_t g0) {
        const int32_t u = (int32_t)(ex - g0);
        const uint32_t before = (uint32_t)__builtin_popcountll(ballot(u < 0));
        tab[lane] = 0u;
        if (u >= 0 && u < 64) __hip_atomic_fetch_max(&tab[u], (uint32_t)lane + 1u, __ATOMIC_RELAXED,
                                                    __HIP_MEMORY_SCOPE_WORKGROUP);
        wave_sync();
        uint32_t x = tab[lane];
        x = scan_max(x > before ? x : before);
        return x - 1u;
    }

    // Copies the runs of the lanes with cnt > 0 (v: virtual position, n:
    // length, s: source -- stage offset of a literal run, offset of a
    // match), all runs of a kind at once.
    template <bool MATCH>
    __device__ __forceinline__ void run_pass(uint32_t v, uint32_t n, uint32_t s, bool on, int32_t rlo) {
        const uint32_t cnt = on && n > 0 ? ((v + n + 15u) >> 4) - (v >> 4) : 0u;
        const uint32_t incl = scan_add(cnt);
        const uint32_t total = rdl(incl, 63);
        const uint32_t ex = incl - cnt;
        for (uint32_t g0 = 0; g0 < total; g0 += 64) {
            const uint32_t gl = g0 + 63 < total ? g0 + 63 : total - 1;
            // runs of the first and last chunk of the pass
            const uint32_t rf = 63u - (uint32_t)__builtin_clzll(ballot(ex <= g0));
            const uint32_t rl = 63u - (uint32_t)__builtin_clzll(ballot(ex <= gl));
            uint32_t rv, rn, rs, rex;
            if (rf == rl) {
                rv = rdl(v, rf);
                rn = rdl(n, rf);
                rs = rdl(s, rf);
                rex = rdl(ex, rf);
            } else {
                const uint32_t r = lane_run(ex, g0);
                rv = bperm(v, r);
                rn = bperm(n, r);
                rs = bperm(s, r);
                rex = bperm(ex, r);
            }
            const uint32_t g = g0 + (uint32_t)lane;
            if (g < total) {
                if constexpr (MATCH)
                    match_chunk<-1>(rv, rn, rs, g - rex, rlo);
                else
                    lit_chunk(rv, rn, rs, g - rex);
            }
            wave_sync();
        }
    }

    // ------------------------------------------------ short sequences
    // Bytes from a token to the next when its match length has no extension
    // and its literal length at most one byte (next: the byte after the
    // token), else 0.
    __device__ __forceinline__ static uint32_t short_dist(uint32_t token, uint32_t next) {
        const uint32_t k = token >= 0xf0u ? 19u + next : (token >> 4) + 3u;
        return (token & 15u) == 15u || (token >= 0xf0u && next == 255u) ? 0u : k;
    }
    // Whether a walk starts at token t2 & 255 (t2 >> 8: the byte after it),
    // `room` bytes before the walk's end: a short sequence of at most 48
    // bytes.  Longer ones, one or two to a window of 256, are parsed faster
    // one at a time (a Llama-3-8B layer of retention 0.24 209 -> 203 us).
    __device__ __forceinline__ static bool walkable(uint32_t t2, uint32_t room) {
        if ((t2 & 15u) == 15u) return false;
        const uint32_t k = short_dist(t2 & 0xffu, (t2 >> 8) & 0xffu);
        return k - 1u < 48u && k <= room;
    }
    // Finds the tokens of a run of such sequences from stage offset x0 on,
    // each next token at or before stage offset xe and no window past x_max:
    // their distances go to the list, their number is returned.
    //
    // The chain of headers is serial; what each link costs is kept small.
    // 256 stage bytes at a time, register r of lane l holds where the next
    // token is if one starts at byte 64 r + l (a multiple of 64 first), so a
    // sequence is one readlane by the position itself and a bit set in a
    // scalar mask; the distances then go to the list 64 at a time.
    __device__ __forceinline__ uint32_t walk(uint32_t x, uint32_t xe, uint32_t x_max) {
        constexpr uint32_t kStop = 0xffffu;  // no short sequence here
        uint32_t n = 0;
        list = 0;
        bool on = true;
        while (on && n + 96u <= kList && x <= x_max) {
            const uint32_t wb = x & ~63u;
            uint32_t nx[4];
#pragma unroll
            for (uint32_t r = 0; r < 4; r++) {
                const uint32_t p = wb + 64u * r + (uint32_t)lane;
                const uint32_t a = p < xe ? p : 0u;
                const uint32_t k = short_dist(stage[a], stage[a + 1u]);
                nx[r] = k - 1u < 255u && p + k <= xe ? p + k : kStop;
            }
            uint64_t mask[4];
            uint32_t o = x, last = x;
#pragma unroll
            for (uint32_t r = 0; r < 4; r++) {
                const uint32_t lim = wb + 64u * (r + 1u);
                uint64_t m = 0;
                while (o < lim) {
                    last = o;
                    m |= 1ull << (o & 63u);
                    o = rdl(nx[r], o & 63u);
                    if (o >= lim) break;
                    last = o;
                    m |= 1ull << (o & 63u);
                    o = rdl(nx[r], o & 63u);
                }
                mask[r] = m;
            }
            if (o == kStop) {
                const uint64_t keep = ~(1ull << (last & 63u));
#pragma unroll
                for (uint32_t r = 0; r < 4; r++)
                    if ((last - wb) >> 6 == r) mask[r] &= keep;
                o = last;
                on = false;
            }
            x = o;
#pragma unroll
            for (uint32_t r = 0; r < 4; r++) {
                // the entries go to lanes n, n + 1, ... (mod 64), a zero from
                // every other lane to the lanes left
                const uint32_t c = (uint32_t)__builtin_popcountll(mask[r]);
                const uint32_t below = __builtin_amdgcn_mbcnt_hi((uint32_t)(mask[r] >> 32),
                                                                 __builtin_amdgcn_mbcnt_lo((uint32_t)mask[r], 0u));
                const bool in = (mask[r] >> lane) & 1ull;
                const uint32_t at = n + (in ? below : c + (uint32_t)lane - below);
                const uint32_t k = nx[r] - (wb + 64u * r + (uint32_t)lane);
                list |= (uint32_t)__builtin_amdgcn_ds_permute((int)(4u * at), in ? (int)(k << (8u * (at >> 6))) : 0);
                n += c;
            }
        }
        return n;
    }

    // Each lane's literal run (n <= kShortLit bytes at stage offset src) to
    // virtual position v, four bytes at a time.
    __device__ __forceinline__ void lit_short(uint32_t v, uint32_t n, uint32_t src) const {
        const lds32 *q = reinterpret_cast<const lds32 *>(stage + (src & ~3u));
        const uint32_t sh = src & 3u;
        uint32_t d0 = n > 0 ? q[0] : 0u;
        for (uint32_t t = 0; ballot(t < n); t += 4) {
            if (t < n) {
                q++;
                const uint32_t d1 = q[0];
                const uint32_t w = __builtin_amdgcn_alignbyte(d1, d0, sh);
                d0 = d1;
#pragma unroll
                for (uint32_t i = 0; i < 4; i++)
                    if (t + i < n) ring[(v + t + i) & kRM] = (uint8_t)(w >> (8 * i));
            }
        }
    }

    // The sources of the lanes' far matches (before rlo, in the written-out
    // output), loaded as dwords: 9 bytes from any position.
    struct FarSrc {
        uint32_t d[3];
    };
    __device__ __forceinline__ uint32_t out_dword(int32_t w) const {
        const int32_t lo = (int32_t)(a0 & ~3u), hi = (int32_t)((a0 + cap - 1u) & ~3u);
        w = w < lo ? lo : w > hi ? hi : w;
        return *reinterpret_cast<const uint32_t *>(obase + w);
    }

    // The batch's matches (lane: n <= kShortMatch bytes at virtual position v,
    // offset off), in rounds: the output bytes of the matches not yet copied
    // are marked in the table, and every match whose source bytes are clear of
    // them copies, one lane each.  The first match left is always clear, so a
    // round copies at least one; sources in the batch rarely chain more than a
    // few deep.  vb: the batch's first virtual position.
    __device__ __forceinline__ void match_short(uint32_t v, uint32_t n, uint32_t off, int32_t rlo, uint32_t vb,
                                                const FarSrc &fs) const {
        const bool live = n > 0;
        const uint32_t r = live ? v - vb : 0u;
        const uint64_t own = live ? ((1ull << n) - 1ull) << (r & 31u) : 0ull;
        const uint32_t ow = r >> 5;
        tab[lane] = 0u;
        if (kTabWords > 64u && lane < (int)(kTabWords - 64u)) tab[64 + lane] = 0u;
        wave_sync();
        if (live) __hip_atomic_fetch_or(&tab[ow], (uint32_t)own, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (own >> 32)
            __hip_atomic_fetch_or(&tab[ow + 1], (uint32_t)(own >> 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        wave_sync();
        // the source's part in this batch
        const int32_t ss = (int32_t)(v - off), rs = ss - (int32_t)vb;
        const int32_t re = rs + (int32_t)(off < n ? off : n);
        const uint32_t cs = rs > 0 ? (uint32_t)rs : 0u;
        const uint64_t need = live && re > 0 ? ((1ull << ((uint32_t)re - cs)) - 1ull) << (cs & 31u) : 0ull;
        const uint32_t nw = need ? cs >> 5 : 0u;
        const bool far = !LDS && ss < rlo, slow = n < 4u || n > 8u || off < n;
        uint64_t pend = ballot(live);
        while (pend) {
            const uint64_t w = ((uint64_t)tab[nw + 1] << 32) | tab[nw];
            const bool go = ((pend >> lane) & 1ull) && (w & need) == 0;
            pend &= ~ballot(go);
            if (go && !slow) {
                // 4 to 8 bytes, not periodic: three dwords hold them
                uint32_t d[3];
#pragma unroll
                for (int i = 0; i < 3; i++)
                    d[i] = *reinterpret_cast<const lds32 *>(ring + ((((uint32_t)ss & ~3u) + 4u * i) & kRM));
                if (!LDS) {
#pragma unroll
                    for (int i = 0; i < 3; i++) d[i] = far ? fs.d[i] : d[i];
                }
                const uint32_t x = __builtin_amdgcn_alignbyte(d[1], d[0], (uint32_t)ss & 3u);
#pragma unroll
                for (uint32_t i = 0; i < 4; i++) ring[(v + i) & kRM] = (uint8_t)(x >> (8 * i));
                if (n > 4u) {
                    const uint32_t y = __builtin_amdgcn_alignbyte(d[2], d[1], (uint32_t)ss & 3u);
#pragma unroll
                    for (uint32_t i = 0; i < 4; i++)
                        if (4u + i < n) ring[(v + 4u + i) & kRM] = (uint8_t)(y >> (8 * i));
                }
            }
            if (go && slow) {
                // byte t from source byte t mod off
                uint32_t m = 0;
                for (uint32_t t = 0; t < n; t++) {
                    uint32_t b;
                    if (far) {
                        const uint32_t w = out_dword((ss + (int32_t)t) & ~3);
                        b = w >> (8u * ((uint32_t)(ss + (int32_t)t) & 3u));
                    } else {
                        b = ring[((uint32_t)ss + m) & kRM];
                    }
                    ring[(v + t) & kRM] = (uint8_t)b;
                    m = m + 1u == off ? 0u : m + 1u;
                }
            }
            wave_sync();
            if (pend && go) {
                __hip_atomic_fetch_and(&tab[ow], ~(uint32_t)own, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                if (own >> 32)
                    __hip_atomic_fetch_and(&tab[ow + 1], ~(uint32_t)(own >> 32), __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_WORKGROUP);
            }
            wave_sync();
        }
    }

    // Copies one parsed batch: lane i < nsl holds slot i (a literal run of
    // ll bytes at stage offset ls, then a match of ml bytes at offset mo);
    // the batch starts at output position op_b and ends at op.
    // ------------------------------------------------ serial copies (long runs)
    // One run at a time in output order, 64 chunks per pass: a chunk's
    // bytes before the run keep what the ring holds (read back), its bytes
    // past the run are don't-care (the next run's first chunk overwrites
    // them; the flush writes out complete chunks only, and a batch ends 32
    // bytes short of the ring slots a near source occupies).
    __device__ __forceinline__ void keep_front(uint32_t cv, uint32_t v, u32x4 &o) const {
        if (cv < v) {  // the run's first chunk: keep its bytes before v
            const u32x4 old = *reinterpret_cast<const ldsx4 *>(ring + (cv & kRM));
#pragma unroll
            for (uint32_t i = 0; i < 4; i++) {
                const uint32_t m = dword_mask(0, v - cv, i);
                o[i] = (old[i] & m) | (o[i] & ~m);
            }
        }
    }
    __device__ __forceinline__ void lit_serial(uint32_t v, uint32_t n, uint32_t src) {
        const uint32_t c0 = v & ~15u;
        const uint32_t nch = ((v + n + 15u) >> 4) - (v >> 4);
        for (uint32_t b = 0; b < nch; b += 64) {
            const uint32_t c = b + (uint32_t)lane;
            if (c < nch) {
                const uint32_t cv = c0 + 16u * c;
                const int32_t sp = (int32_t)(src + cv - v);
                const lds32 *q = reinterpret_cast<const lds32 *>(stage + (sp & ~3));
                uint32_t d[5];
#pragma unroll
                for (int i = 0; i < 5; i++) d[i] = q[i];
                u32x4 o = realign(d, (uint32_t)sp & 3u);
                keep_front(cv, v, o);
                *reinterpret_cast<ldsx4 *>(ring + (cv & kRM)) = o;
            }
            wave_sync();
        }
    }
    template <int K>
    __device__ __forceinline__ void match_serial(uint32_t v, uint32_t n, uint32_t off, int32_t rlo) {
        const uint32_t c0 = v & ~15u;
        const uint32_t nch = ((v + n + 15u) >> 4) - (v >> 4);
        for (uint32_t b = 0; b < nch; b += 64) {
            const uint32_t c = b + (uint32_t)lane;
            if (c < nch) {
                const uint32_t cv = c0 + 16u * c;
                const int32_t r0 = (int32_t)(cv - v);
                u32x4 o;
                if (K == 0) {
                    o = src16((int32_t)(cv - off), rlo);
                } else if (K == 1) {
                    const uint32_t a = umod((uint32_t)(r0 + (int32_t)off), off);
                    const int32_t base = (int32_t)(v - off + a);
                    o = src16(base, rlo);
                    const u32x4 bb = src16(base - (int32_t)off, rlo);
                    const uint32_t kw = off - a < 16u ? off - a : 16u;
#pragma unroll
                    for (uint32_t i = 0; i < 4; i++) {
                        const uint32_t m = dword_mask(0, kw, i);
                        o[i] = (o[i] & m) | (bb[i] & ~m);
                    }
                } else {
                    uint32_t m = umod((uint32_t)(r0 + 16 * (int32_t)off), off);
                    const uint32_t sv = v - off;
                    uint32_t dd[4] = {0u, 0u, 0u, 0u};
#pragma unroll
                    for (uint32_t t = 0; t < 16; t++) {
                        dd[t >> 2] |= (uint32_t)ring[(sv + m) & kRM] << (8 * (t & 3));
                        m = m + 1 == off ? 0u : m + 1;
                    }
                    o = u32x4{dd[0], dd[1], dd[2], dd[3]};
                }
                keep_front(cv, v, o);
                *reinterpret_cast<ldsx4 *>(ring + (cv & kRM)) = o;
            }
            wave_sync();
        }
    }

    __device__ __forceinline__ void execute(uint32_t nsl, uint32_t op_b, uint32_t ls, uint32_t ll, uint32_t mo,
                                            uint32_t ml) {
        const bool live = (uint32_t)lane < nsl;
        ll = live ? ll : 0u;
        ml = live ? ml : 0u;
        const uint32_t len = ll + ml;
        const uint32_t vl = op_b + a0 + scan_add(len) - len;  // virtual start of the slot
        const uint32_t vm = vl + ll;
        // The ring's slots from the batch's end on hold the R bytes before it,
        // but up to 15 of them may be the don't-care bytes of a long run's
        // last chunk, in an earlier batch too when this one is shorter than
        // that: the ring serves sources from rlo on, 32 bytes after its
        // start, and what lies before is in the written-out output.
        const int32_t rlo = (int32_t)(op + a0) - (int32_t)R + 32;
        // Long runs one per pass: 128 bytes each on average or, where every
        // match is short (and shares a pass with others), literals of about
        // 640.  Sparse tiles' blocks hold such: at 256 for both a fused layer
        // of hidden size 512 and retention 0.21 took 73 us, now 63; half-zeroed
        // data with long matches 49 us (600 blocks of 16 KiB) at 640, 44 at 256.
        const bool tiny_m = ballot(ml > kShortMatch) == 0;
        if (op - op_b >= (tiny_m ? 640u : 256u) * nsl) {
            for (uint32_t i = 0; i < nsl; i++) {
                const uint32_t v = rdl(vl, i), n = rdl(ll, i);
                if (n > 0) lit_serial(v, n, rdl(ls, i));
                const uint32_t m = rdl(ml, i);
                if (m > 0) {
                    const uint32_t off = rdl(mo, i);
                    if (off >= m)
                        match_serial<0>(v + n, m, off, rlo);
                    else if (off >= 16u)
                        match_serial<1>(v + n, m, off, rlo);
                    else
                        match_serial<2>(v + n, m, off, rlo);
                }
            }
            return;
        }
        // short runs: all literal runs of the batch at once, then the matches
        const bool short_m = tiny_m && op - op_b <= kShortBytes;
        FarSrc fs;
        if (short_m && !LDS) {
            // far sources are final: their loads run beside the literal copies
            const int32_t ss = (int32_t)(vm - mo);
            if (ml > 0 && ss < rlo) {
#pragma unroll
                for (int i = 0; i < 3; i++) fs.d[i] = out_dword((ss & ~3) + 4 * i);
            }
        }
        if (ballot(ll > kShortLit) == 0) {
            lit_short(vl, ll, ls);
            wave_sync();
        } else {
            run_pass<false>(vl, ll, ls, live, rlo);
        }
        if (short_m) {
            match_short(vm, ml, mo, rlo, op_b + a0, fs);
            return;
        }
        // matches in order; a pass takes the next pending match and every
        // following one up to the first whose source reaches past the start
        // of that first match
        const int32_t src_hi = (int32_t)(vm - mo + (mo < ml ? mo : ml));
        uint64_t pend = ballot(live && ml > 0);
        while (pend) {
            const uint32_t j0 = (uint32_t)__builtin_ctzll(pend);
            const int32_t D = (int32_t)rdl(vm, j0);
            const uint64_t block = pend & ~ballot(src_hi <= D);
            const uint64_t upto = block >> j0 ? ((1ull << ((uint32_t)__builtin_ctzll(block >> j0) + j0)) - 1) : ~0ull;
            const uint64_t grp = pend & upto;
            if ((grp & (grp - 1)) == 0) {
                // one match: its chunks over the lanes
                const uint32_t v = rdl(vm, j0), n = rdl(ml, j0), off = rdl(mo, j0);
                const uint32_t nch = ((v + n + 15u) >> 4) - (v >> 4);
                for (uint32_t c0 = 0; c0 < nch; c0 += 64) {
                    const uint32_t c = c0 + (uint32_t)lane;
                    if (c < nch) {
                        if (off >= n)
                            match_chunk<0>(v, n, off, c, rlo);
                        else if (off >= 16u)
                            match_chunk<1>(v, n, off, c, rlo);
                        else
                            match_chunk<2>(v, n, off, c, rlo);
                    }
                    wave_sync();
                }
            } else {
                run_pass<true>(vm, ml, mo, ((grp >> lane) & 1ull) != 0, rlo);
            }
            pend &= ~grp;
        }
    }

    // Writes the output [fl, op) out: all of it when `exact`, else up to the
    // last 16-aligned virtual position.
    __device__ __forceinline__ void flush(bool exact) {
        if constexpr (LDS) {
            fl = op;
            return;
        }
        const uint32_t vf = fl + a0, vo = op + a0;
        const uint32_t ve = exact ? vo : (vo & ~15u);
        if (ve <= vf) return;
        uint32_t h = (16u - (vf & 15u)) & 15u;
        if (h > ve - vf) h = ve - vf;
        if (lane < (int)h) obase[vf + lane] = ring[(vf + lane) & kRM];
        const uint32_t vb = vf + h;
        const uint32_t nch = (ve - vb) >> 4;
        for (uint32_t c = lane; c < nch; c += 64) {
            const uint32_t x = vb + 16u * c;
            *reinterpret_cast<u32x4 *>(obase + x) = *reinterpret_cast<const ldsx4 *>(ring + (x & kRM));
        }
        const uint32_t vt = vb + 16u * nch;
        if (lane < (int)(ve - vt)) obase[vt + lane] = ring[(vt + lane) & kRM];
        fl = ve - a0;
        __asm__ __volatile__("" ::: "memory");
    }
};

// Decodes one block whose input is [0, ilen) (block-relative) into d; on
// return code / detail / pos / req hold the outcome (HH_OK or the
// reference's error record) and d.op the bytes decoded.  The caller writes
// out the rest of a successful block (d.flush(true)).  `staged`: the caller
// has already put the stage for input position 0 in place.
//
// A batch is parsed in three ways.  Runs of short sequences come from a walk
// over their tokens (SeqDec::walk), each lane then reading its sequence's
// fields; between them the fast loop follows the chain of headers -- token,
// literal length, offset, match length -- and records each sequence in a
// lane, stopping where a header would leave the stage or a length extension
// is longer than 7 (6) bytes.  The wave then checks all of the recorded
// sequences at once (input bounds, capacity, offsets, the batch budget) and
// keeps those before the first one that fails.  The general step parses the sequence after them one state at a time with
// every check in the reference's order: a run continued from the previous
// batch, a run cut by the stage end or the budget, long extensions, and
// every error, reported as the reference reports it.
template <uint32_t R, uint32_t S, bool LDS, typename Progress = NoProgress>
__device__ __forceinline__ void decode_block(SeqDec<R, S, LDS> &d, uint32_t ilen, int32_t &code, int32_t &detail,
                                             uint64_t &pos, uint64_t &req, bool staged = false,
                                             Progress &&progress = Progress{}) {
    using D = SeqDec<R, S, LDS>;
    const uint32_t end = ilen;
    const uint32_t cap = d.cap;
    const uint32_t lane = (uint32_t)d.lane;
    uint32_t ip = 0;
    uint32_t ms = kToken;
    uint32_t lit_rem = 0, m_rem = 0, m_off = 0, tml = 0;
    uint64_t acc = 0;  // kLitExt, kMatchExt: the length so far
    d.hv = 0;
    d.hb = 0;
    d.list = 0;
    // the list of short sequences: next entry (the one at ip), entries
    uint32_t li = 0, ln = 0;
    d.pf_on = false;
    if (end == 0) return;
    if (!staged)
        d.restage(0);
    else
        d.prefetch();
    for (;;) {
        // ---------------------------------------------------------- parse
        const uint32_t op_b = d.op;
        uint32_t op = d.op;
        uint32_t nsl = 0, bout = 0;
        // the batch's output may not pass lim (near match sources stay in
        // the ring)
        uint32_t lim = 0xffffffffu;
        bool done = false, restage = false;
        // slots in lanes (slot i in lane i): literal stage offset and length,
        // match offset and length, token position (fast loop only)
        uint32_t ls = 0, ll = 0, mo = 0, ml = 0, tp = 0;
        bool walked = false;  // the slot is a sequence from the list
        if (ms != kToken) nsl = 1;  // a run continued from the previous batch
        for (;;) {
            // ---- fast loop: header chain only
            if (ms == kToken) {
                const uint32_t f0 = nsl;
                // last position a header may start at: before the block end,
                // with 8 bytes in the stage
                const uint32_t hl = d.at_end ? end - 1u : (end - 1u < d.sb + (S - 8u) ? end - 1u : d.sb + (S - 8u));
                uint32_t fp = ip;
                // output end and near-match limit of the chain so far: the
                // loop stops before a sequence that would pass the batch's
                // budget or limit (the check after it then rarely fails)
                uint32_t fo = op;
                uint32_t fl = lim < op_b + D::kOB ? lim : op_b + D::kOB;
                bool full = false;
                uint32_t lt = 0;  // how many of the last slots came from the list
                // short sequences end inside the stage and the block
                const uint32_t we = d.at_end || end - d.sb < S ? end - d.sb : S;
                for (;;) {
                    // short sequences, up to 64 at once from the list
                    const uint32_t w0 = nsl;
                    if (nsl < 64u && fp <= hl && fo < fl) {
                        if (li == ln) {
                            if (!d.in_win8(fp)) d.read16(fp);
                            if (D::walkable((uint32_t)d.peek8(fp), we - (fp - d.sb))) {
                                // (their output is at least their input: no
                                // token past the batch's budget)
                                ln = d.walk(fp - d.sb, we, fp - d.sb + (fl - fo));
                                li = 0;
                            }
                        }
                        if (li < ln) {
                            const uint32_t n = ln - li < 64u - nsl ? ln - li : 64u - nsl;
                            const bool me = lane >= w0 && lane < w0 + n;
                            const uint32_t e = li + lane - w0;
                            const uint32_t kw = bperm(d.list, e) >> (8u * ((e >> 6) & 3u));
                            const uint32_t k = me ? kw & 0xffu : 0u;
                            const uint32_t ke = scan_add(k);
                            if (me) {
                                tp = fp - d.sb + ke - k;
                                const uint32_t token = d.stage[tp], next = d.stage[tp + 1u];
                                const bool x1 = token >= 0xf0u;
                                ls = tp + (x1 ? 2u : 1u);
                                ll = x1 ? 15u + next : token >> 4;
                                ml = (token & 15u) + 4u;
                                mo = (uint32_t)d.stage[ls + ll] | ((uint32_t)d.stage[ls + ll + 1u] << 8);
                                tp += d.sb;
                                walked = true;
                            }
                            fo += rdl(scan_add(me ? ll + ml : 0u), 63);
                            lt = n;
                            li += n;
                            nsl += n;
                            fp += rdl(ke, 63);
                        }
                    }
                    // then the others, one at a time, until a short one
                    // follows
                    bool back = false, any = false;
                    while (nsl < 64u && fp <= hl) {
                        if (!d.in_win8(fp)) d.read16(fp);
                        const uint64_t t8 = d.peek8(fp);
                        const uint32_t token = (uint32_t)t8 & 0xffu;
                        uint32_t lit = token >> 4;
                        if (any && fo < fl && D::walkable((uint32_t)t8, we - (fp - d.sb))) {
                            back = true;
                            break;
                        }
                        any = true;
                        uint32_t p = fp + 1;
                        if (lit == 15u) {
                            const uint64_t x = t8 >> 8;
                            const uint32_t e = (uint32_t)__builtin_ctzll(~x | (1ull << 56)) >> 3;  // 7: none
                            if (e == 7u) break;
                            lit += 255u * e + (uint32_t)((x >> (8 * e)) & 0xffu);
                            p += e + 1;
                        }
                        const uint32_t le = p + lit;  // offset position
                        if (le > hl) break;
                        if (!d.in_win8(le)) d.read16(le);
                        const uint64_t o8 = d.peek8(le);
                        uint32_t mlen = (token & 15u) + 4u;
                        uint32_t q = le + 2;
                        if ((token & 15u) == 15u) {
                            const uint64_t x = o8 >> 16;
                            const uint32_t e = (uint32_t)__builtin_ctzll(~x | (1ull << 48)) >> 3;  // 6: none
                            if (e == 6u) break;
                            mlen += 255u * e + (uint32_t)((x >> (8 * e)) & 0xffu);
                            q += e + 1;
                        }
                        const uint32_t off = (uint32_t)o8 & 0xffffu;
                        const uint32_t fm = fo + lit;
                        uint32_t fl2 = fl;
                        if (!LDS && off <= R - 128u && off <= fm) {
                            const uint32_t l2 = fm - off + (R - 64u);
                            fl2 = l2 < fl2 ? l2 : fl2;
                        }
                        if (fm + mlen > fl2) {
                            full = true;
                            break;
                        }
                        const bool me = lane == nsl;
                        tp = me ? fp : tp;
                        ls = me ? p - d.sb : ls;
                        ll = me ? lit : ll;
                        mo = me ? off : mo;
                        ml = me ? mlen : ml;
                        nsl++;
                        lt = 0;
                        fp = q;
                        fo = fm + mlen;
                        fl = fl2;
                    }
                    if (!back) break;
                }
                if (nsl > f0) {
                    // check slots f0 .. nsl - 1 at once; keep those before
                    // the first that fails (the general step parses it again)
                    const bool live = lane < nsl;
                    const uint32_t len = live ? ll + ml : 0u;
                    const uint32_t oe = op_b + scan_add(len);  // output end of each slot
                    const uint32_t om = oe - ml;               // output position of the match
                    const uint32_t qn = bperm(tp, lane + 1u);
                    const uint32_t q = lane + 1u == nsl ? fp : qn;  // input end of each slot
                    // near-match limit: prefix minimum over the fast slots
                    // (a walked sequence's match does not end the batch for a
                    // source that leaves the ring: it reads the output)
                    uint32_t nl = (!LDS && lane >= f0 && live && mo <= R - 128u && !walked)
                                      ? om - mo + (R - 64u)
                                      : 0xffffffffu;
                    nl = ~scan_max(~nl);
                    nl = nl < lim ? nl : lim;
                    const bool valid = q <= end && om < cap && mo != 0u && mo <= om && oe <= cap;
                    const bool ok = valid && oe - op_b <= D::kOB && oe <= nl;
                    const uint64_t badm = ballot(!ok && lane >= f0 && live);
                    const uint32_t f = badm ? (uint32_t)__builtin_ctzll(badm) : nsl;
                    if (f > f0) {
                        op = rdl(oe, f - 1u);
                        lim = rdl(nl, f - 1u);
                        bout = op - op_b;
                    }
                    // a slot past the batch's budget or limit starts the next batch
                    if (f < nsl) full = (ballot(valid) >> f) & 1ull;
                    ip = f < nsl ? rdl(tp, f) : fp;
                    // the list goes on with the first slot not kept, if
                    // that came from it
                    if (f < nsl) {
                        const bool listed = nsl - f <= lt;
                        li = listed ? li - (nsl - f) : 0u;
                        ln = listed ? ln : 0u;
                    }
                    nsl = f;
                    const bool keep = lane < f;
                    ls = keep ? ls : 0u;
                    ll = keep ? ll : 0u;
                    mo = keep ? mo : 0u;
                    ml = keep ? ml : 0u;
                }
                // the next sequence does not fit this batch: start the next
                // one with it (the general step splits only a sequence that
                // an empty batch cannot hold)
                if (full && bout > 0) break;
            }
            // ---- general step
            if (ms <= kLitExt) {
                // token and literal length (block.rs:270-289); the extension
                // bytes usually lie in the 7 bytes after the token
                uint32_t p = ip;
                uint64_t lit;
                bool ext = true;
                if (ms == kToken) {
                    if (ip >= end) {
                        done = true;
                        break;
                    }
                    if (nsl == 64u) break;
                    if (!d.in_win8(ip) && !d.in_stage8(ip)) {
                        restage = true;
                        break;
                    }
                    const uint64_t t8 = d.get8(ip);
                    const uint32_t token = (uint32_t)t8 & 0xffu;
                    tml = token & 15u;
                    lit = token >> 4;
                    p++;
                    ext = false;
                    if (lit == 15) {
                        const uint64_t x = t8 >> 8;
                        const uint32_t e = (uint32_t)__builtin_ctzll(~x | (1ull << 56)) >> 3;  // 7: none
                        ext = e == 7u;
                        if (!ext && p + e >= end) {
                            code = HH_ERR_UNEXPECTED_EOF;
                            pos = ilen;
                            return;
                        }
                        lit += 255u * e + (ext ? 0u : (uint32_t)((x >> (8 * e)) & 0xffu));
                        p += ext ? 7u : e + 1u;
                    }
                } else {
                    lit = acc;
                }
                if (ext) {
                    const int r = d.ext_slow(p, end, lit);
                    if (r == 1) {
                        code = HH_ERR_UNEXPECTED_EOF;
                        pos = ilen;
                        return;
                    }
                    if (r == 2) {
                        if (bout == 0) {
                            ip = p;
                            acc = lit;
                            ms = kLitExt;
                        }
                        restage = true;
                        break;
                    }
                    // a length beyond 32 bits exceeds the block input:
                    // the input-length check below fails for it too
                    if (lit > 0xffffffffull) {
                        code = HH_ERR_UNEXPECTED_EOF;
                        pos = p;
                        return;
                    }
                }
                lit_rem = (uint32_t)lit;
                if (lit_rem > 0) {
                    if (end - p < lit_rem) {
                        code = HH_ERR_UNEXPECTED_EOF;
                        pos = p;
                        return;
                    }
                    if (lit_rem > cap - op) {
                        code = HH_ERR_BUFFER_TOO_SMALL;
                        req = (uint64_t)op + lit_rem;
                        return;
                    }
                }
                if (ms == kToken) nsl++;  // the sequence's slot (zero in every lane)
                ip = p;
                ms = kLit;
            }
            if (ms == kLit) {
                if (lit_rem > 0) {
                    const uint32_t av = d.lit_avail(ip);
                    uint32_t n = lit_rem < av ? lit_rem : av;
                    if (n > D::kOB - bout) n = D::kOB - bout;
                    if (n > lim - op) n = lim - op;
                    if (n == 0) {
                        restage = av == 0;
                        break;
                    }
                    const bool me = lane == nsl - 1u;
                    ls = me ? ip - d.sb : ls;
                    ll = me ? n : ll;
                    ip += n;
                    op += n;
                    bout += n;
                    lit_rem -= n;
                    if (lit_rem > 0) {
                        restage = av == n;
                        break;
                    }
                }
                if (op >= cap) {  // block.rs:309-311
                    done = true;
                    break;
                }
                ms = kOff;
            }
            if (ms == kOff || ms == kMatchExt) {
                // offset and match length (block.rs:313-345)
                uint32_t p = ip;
                uint64_t mlen;
                bool ext = true;
                if (ms == kOff) {
                    if (end - ip < 2) {
                        code = HH_ERR_UNEXPECTED_EOF;
                        pos = ip;
                        return;
                    }
                    if (!d.in_win8(ip) && !d.in_stage8(ip)) {
                        restage = true;
                        break;
                    }
                    const uint64_t o8 = d.get8(ip);
                    m_off = (uint32_t)o8 & 0xffffu;
                    p += 2;
                    if (m_off == 0) {
                        code = HH_ERR_CORRUPTED_DATA;
                        detail = HH_CORRUPT_ZERO_OFFSET;
                        return;
                    }
                    if (m_off > op) {
                        code = HH_ERR_CORRUPTED_DATA;
                        detail = HH_CORRUPT_OFFSET_BEYOND;
                        pos = op;
                        return;
                    }
                    mlen = tml + 4u;
                    ext = false;
                    if (tml == 15u) {
                        const uint64_t x = o8 >> 16;
                        const uint32_t e = (uint32_t)__builtin_ctzll(~x | (1ull << 48)) >> 3;  // 6: none
                        ext = e == 6u;
                        if (!ext && p + e >= end) {
                            code = HH_ERR_UNEXPECTED_EOF;
                            pos = ilen;
                            return;
                        }
                        mlen += 255u * e + (ext ? 0u : (uint32_t)((x >> (8 * e)) & 0xffu));
                        p += ext ? 6u : e + 1u;
                    }
                } else {
                    mlen = acc;
                }
                if (ext) {
                    const int r = d.ext_slow(p, end, mlen);
                    if (r == 1) {
                        code = HH_ERR_UNEXPECTED_EOF;
                        pos = ilen;
                        return;
                    }
                    if (r == 2) {
                        if (bout == 0) {
                            ip = p;
                            acc = mlen;
                            ms = kMatchExt;
                        }
                        restage = true;
                        break;
                    }
                    if (mlen > 0xffffffffull) {  // more than any capacity
                        code = HH_ERR_BUFFER_TOO_SMALL;
                        req = (uint64_t)op + mlen;
                        return;
                    }
                }
                if (mlen > cap - op) {
                    code = HH_ERR_BUFFER_TOO_SMALL;
                    req = (uint64_t)op + mlen;
                    return;
                }
                ip = p;
                m_rem = (uint32_t)mlen;
                ms = kMatch;
            }
            // ms == kMatch: a match whose offset fits the ring reads it
            // there: the batch then ends before its output reaches R - 64
            // bytes past the match's source
            uint32_t lm = lim;
            if (!LDS && m_off <= R - 128u) {
                const uint32_t l2 = op - m_off + (R - 64u);
                lm = l2 < lm ? l2 : lm;
            }
            uint32_t n = m_rem;
            if (n > D::kOB - bout) n = D::kOB - bout;
            if (n > lm - op) n = lm - op;
            if (n == 0) break;
            lim = lm;
            {
                const bool me = lane == nsl - 1u;
                mo = me ? m_off : mo;
                ml = me ? n : ml;
            }
            op += n;
            bout += n;
            m_rem -= n;
            if (m_rem > 0) break;
            ms = kToken;
        }
        // ---------------------------------------------------------- copy
        // the next stage is put in place after the copies (which read the
        // current one) and before the batch's output is written out, so the
        // wait for its loads does not include those stores (a wave's memory
        // operations complete in order)
        d.op = op;
        if (bout > 0) d.execute(nsl, op_b, ls, ll, mo, ml);
        if (restage) {
            d.restage(ip);
            li = ln = 0;
        }
        if (bout > 0) {
            d.flush(false);
            progress(op);
        }
        if (done) return;
    }
}

}  // namespace seq
}  // namespace hh

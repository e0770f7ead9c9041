// mfma_tiles.hpp — what the matrix-core products share: the split of fp32 activations
// into two fp16 parts, the decode of packed weights to exact fp16 MFMA operands and the
// byte layout of staged weight rows (grouped.hip, wide.hip).
#pragma once

#include "device_common.hpp"
#include "gemv_stream.hpp"
#include "host_common.hpp"
#include "kernels.hpp"
#include "quant_rules.hpp"
#include "swiglu.hpp"

namespace objeta {
namespace dev {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr uint32_t kPerm[8] = {0, 4, 1, 5, 2, 6, 3, 7};
constexpr uint32_t kSlab = 16;  // rows of one MFMA tile

// The power of two 2^s that brings a row of maximum magnitude m below 2^14 (s = 0
// for a zero or non-finite row).
__device__ __forceinline__ int split_shift(float m) {
    int s = 0;
    if (m > 0.0f && __builtin_isfinite(m)) {
        int ex;
        (void)frexpf(m, &ex);  // m < 2^ex
        s = 14 - ex;
        s = s > 126 ? 126 : s;  // 2^-s stays a normal float
    }
    return s;
}

// ------------------------------------------------------------- split rows
// One workgroup per row: scale = 2^s with |x 2^s| < 2^14, then hi = fp16(x 2^s),
// lo = fp16(x 2^s - hi), stored in the (w0,w4),(w1,w5),.. order of each group of
// 8 when perm is set, else in element order; mult[row] = 2^-s restores the
// products. s comes from the finite elements; an infinity or NaN is its own hi part
// (lo 0), so it propagates as in a plain product. lo may be NULL (hi alone).
__device__ inline void split_row(const float* __restrict__ src, uint32_t cols, _Float16* __restrict__ hi,
                          _Float16* __restrict__ lo, float* __restrict__ mult, uint32_t row, uint32_t perm) {
    __shared__ float red[4];
    const float* x = src + static_cast<size_t>(row) * cols;
    float m = 0.0f;
    for (uint32_t c = threadIdx.x; c < cols; c += 256) {
        const float v = x[c];
        m = __builtin_isfinite(v) ? fmaxf(m, fabsf(v)) : m;
    }
    for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    const int s = split_shift(m);
    if (threadIdx.x == 0) mult[row] = ldexpf(1.0f, -s);
    _Float16* h = hi + static_cast<size_t>(row) * cols;
    _Float16* l = lo + static_cast<size_t>(row) * cols;
    for (uint32_t g = threadIdx.x; g < cols / 8; g += 256) {
        const float4 a = *reinterpret_cast<const float4*>(x + 8 * g);
        const float4 b = *reinterpret_cast<const float4*>(x + 8 * g + 4);
        const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
        half8 vh, vl;
#pragma unroll
        for (int d = 0; d < 8; ++d) {
            const float xs = ldexpf(v[perm ? kPerm[d] : d], s);
            const _Float16 th = static_cast<_Float16>(xs);
            vh[d] = th;
            vl[d] = __builtin_isfinite(xs) ? static_cast<_Float16>(xs - static_cast<float>(th)) : static_cast<_Float16>(0.0f);
        }
        *reinterpret_cast<half8*>(h + 8 * g) = vh;
        if (lo) *reinterpret_cast<half8*>(l + 8 * g) = vl;
    }
}

// ------------------------------------------------------ weights -> B operand
// A lane's 8 weights of one block as exact fp16 values in the (w0,w4),(w1,w5),
// (w2,w6),(w3,w7) order of the split activations.
__device__ __forceinline__ half8 pack8(h2 a, h2 b, h2 c, h2 d) {
    half8 r;
    r[0] = a.x; r[1] = a.y; r[2] = b.x; r[3] = b.y;
    r[4] = c.x; r[5] = c.y; r[6] = d.x; r[7] = d.y;
    return r;
}

// The constants of the decodes that v_and_or_b32 takes from a register: an instruction of
// gfx9 reads one scalar constant, so mask and magic together cost a separate and and or
// unless one sits in a vector register (the empty asm hides its value; without side
// effects, it is hoisted out of the loops).
__device__ __forceinline__ uint32_t in_vgpr(uint32_t v) {
    asm("" : "+v"(v));
    return v;
}

// nibble dword n (weights 2m, 2m+1 in byte m), optional 5th bits m8 (bit i: weight i):
// fp16 1024 + q (or 1024 + 16 q) by OR-ing the field into the significand, then the zero
// point taken off. The 5th bits of a pair go 16 apart, then to above their nibble. (The
// products by constants that spread them before are multiplies at a quarter of the rate.) The
// 512-token Q4_0 layer of 128 2048 x 768 experts: 361 -> 353 us.
template <bool Q5>
__device__ __forceinline__ half8 nibbles_to_b(uint32_t n, uint32_t m8) {
    const uint32_t magic = in_vgpr(0x64006400u);
    const uint32_t n8 = n >> 8;
    const _Float16 blo = Q5 ? (_Float16)1040.0f : (_Float16)1032.0f;  // 1024 + zero point
    const _Float16 bhi = Q5 ? (_Float16)-80.0f : (_Float16)-72.0f;    // 64 + zero point
    const h2 klo = {blo, blo}, khi = {bhi, bhi}, k16 = {(_Float16)0.0625f, (_Float16)0.0625f};
    uint32_t a = (n & 0x000F000Fu) | magic, b = (n & 0x00F000F0u) | magic;
    uint32_t c = (n8 & 0x000F000Fu) | magic, d = (n8 & 0x00F000F0u) | magic;
    if constexpr (Q5) {
        const uint32_t h = m8 | (m8 << 12);  // bit i: weight i, bit 16 + i: weight i + 4 (i < 4)
        a |= (h << 4) & 0x00100010u;
        b |= (h << 7) & 0x01000100u;
        c |= (h << 2) & 0x00100010u;
        d |= (h << 5) & 0x01000100u;
    }
    return pack8(as_h2(a) - klo, as_h2(b) * k16 + khi, as_h2(c) - klo, as_h2(d) * k16 + khi);
}

// IQ3_0: 2-bit lows lo16 (weights 8kg .. 8kg+7) and 1-bit highs h8 -> the 8 weights
// q - 4 as exact fp16 in the (w0,w4),(w1,w5),.. order: the lows' bytes and the highs'
// nibbles go 16 apart, a pair's fields stay where they are (q 4^i, exact in the
// significand) and the zero point's multiply-add scales them back. 19 operations instead
// of 40 (8 vectors by 14336 x 4096 21.0 -> 18.0 us, 64 vectors 56.7 -> 52.2).
__device__ __forceinline__ half8 iq3_to_b(uint32_t lo16, uint32_t h8) {
    const uint32_t magic = in_vgpr(0x64006400u);
    const uint32_t e = __builtin_amdgcn_perm(0u, lo16, 0x0C010C00u);  // bytes: lows 0..3, 0, lows 4..7, 0
    const uint32_t h = h8 | (h8 << 12);  // bit i: weight i, bit 16 + i: weight i + 4 (i < 4)
    const h2 k0 = {(_Float16)1028.0f, (_Float16)1028.0f};
    h2 p[4];
    p[0] = as_h2(((e & 0x00030003u) | magic) | ((h << 2) & 0x00040004u)) - k0;
    const _Float16 sc[4] = {(_Float16)1.0f, (_Float16)0.25f, (_Float16)0.0625f, (_Float16)0.015625f};
    const _Float16 zp[4] = {(_Float16)-1028.0f, (_Float16)-260.0f, (_Float16)-68.0f, (_Float16)-20.0f};
#pragma unroll
    for (int i = 1; i < 4; ++i) {
        const uint32_t v = ((e & (0x00030003u << (2 * i))) | magic) | ((h << (i + 2)) & (0x00040004u << (2 * i)));
        p[i] = as_h2(v) * h2{sc[i], sc[i]} + h2{zp[i], zp[i]};
    }
    return pack8(p[0], p[1], p[2], p[3]);
}

// ------------------------------------------------------------- staged tiles
// Staged row segments: weights (and, for the split FP4 layout, the E8M0 scales) of columns
// [c0, c0 + kc). wdw / sdw: dwords of a row segment. kChunkGU / kChunkDn: columns per
// staged chunk of the eight-member sets (grouped.hip), gate and up together / down, the
// widths that measured fastest there; lds_dw: LDS dwords of such a chunk. kTileScale: one E8M0 byte per 128 x 128
// tile (FP8), taken per chunk into a register by tile_scales instead of being staged per
// row.
template <class R>
struct Tile;

template <int F>
struct Tile<QRows<F>> {
    static constexpr int kBB = Fmt<F>::kBlockBytes;
    static constexpr bool kPermuted = true;  // weights in the (w0,w4),(w1,w5),.. order
    static constexpr bool kScales = false;
    static constexpr bool kTileScale = false;
    static constexpr uint32_t kChunkGU = 512, kChunkDn = 256;
    static constexpr __host__ __device__ uint32_t wdw(uint32_t kc) { return kc / 32 * kBB / 4; }  // dwords per row segment
    static constexpr __host__ __device__ uint32_t sdw(uint32_t) { return 0; }
    static constexpr __host__ __device__ uint32_t lds_dw(uint32_t kc) { return kSlab * (wdw(kc) + 4); }
    static __device__ __forceinline__ size_t wpitch(const QRows<F>& m) { return m.row_bytes; }
    static __device__ __forceinline__ size_t spitch(const QRows<F>&) { return 0; }
    static __device__ __forceinline__ const uint8_t* wrow(const QRows<F>& m, uint32_t c0) {
        return m.q + static_cast<size_t>(c0 / 32) * kBB;
    }
    static __device__ __forceinline__ const uint8_t* srow(const QRows<F>&, uint32_t) { return nullptr; }
    static __device__ __forceinline__ uint32_t tile_scales(const QRows<F>&, uint32_t, uint32_t, uint32_t) { return 0; }
    // block b of a row (LDS row base `w`), k group kg: 8 weights and the scale
    static __device__ __forceinline__ half8 get(const uint8_t* w, const uint8_t*, uint32_t, uint32_t b, uint32_t kg,
                                                float& scale) {
        const uint8_t* blk = w + b * kBB;
        auto u16 = [&](uint32_t o) { return static_cast<uint32_t>(*reinterpret_cast<const uint16_t*>(blk + o)); };
        // a dword at 2-byte alignment as two reads (one unaligned LDS read took 14% longer
        // over the whole product, two aligned dwords and a byte shift 1 to 3%)
        auto u32 = [&](uint32_t o) { return u16(o) | (u16(o + 2) << 16); };
        scale = f16_to_f32(u16(0));
        if constexpr (F == kQ4) {
            return nibbles_to_b<false>(u32(2 + 4 * kg), 0);
        } else if constexpr (F == kQ5) {
            return nibbles_to_b<true>(u32(6 + 4 * kg), blk[2 + kg]);
        } else {
            return iq3_to_b(u16(2 + 2 * kg), blk[10 + kg]);
        }
    }
};

template <>
struct Tile<Fp4Rows> {
    static constexpr bool kPermuted = false;
    static constexpr bool kScales = true;
    static constexpr bool kTileScale = false;
    static constexpr uint32_t kChunkGU = 512, kChunkDn = 512;
    static constexpr __host__ __device__ uint32_t wdw(uint32_t kc) { return kc / 8; }   // kc / 2 bytes
    static constexpr __host__ __device__ uint32_t sdw(uint32_t kc) { return kc / 128; }  // kc / 32 bytes (kc % 128 == 0)
    static constexpr __host__ __device__ uint32_t lds_dw(uint32_t kc) {
        return kSlab * (wdw(kc) + 4) + kSlab * (sdw(kc) + 1);
    }
    static __device__ __forceinline__ size_t wpitch(const Fp4Rows& m) { return m.wrow; }
    static __device__ __forceinline__ size_t spitch(const Fp4Rows& m) { return m.srow; }
    static __device__ __forceinline__ const uint8_t* wrow(const Fp4Rows& m, uint32_t c0) { return m.w + c0 / 2; }
    static __device__ __forceinline__ const uint8_t* srow(const Fp4Rows& m, uint32_t c0) { return m.s + c0 / 32; }
    static __device__ __forceinline__ uint32_t tile_scales(const Fp4Rows&, uint32_t, uint32_t, uint32_t) { return 0; }
    // the 8 weights in element order (the hardware conversion's pairs)
    static __device__ __forceinline__ half8 get(const uint8_t* w, const uint8_t* sc, uint32_t, uint32_t b, uint32_t kg,
                                                float& scale) {
        scale = e8m0_to_f32(sc[b]);
        const uint32_t n = *reinterpret_cast<const uint32_t*>(w + 16 * b + 4 * kg);
        h2 p[4];
        fp4_to_h2x4(n, p);
        return pack8(p[0], p[1], p[2], p[3]);
    }
};

// FP8 E4M3 rows ([rows][cols] bytes) with an E8M0 byte per 128 x 128 tile. A code
// decodes by the reference's rule (rules::f8e4m3_to_f32: exponent field 0 as
// mant * 2^-5, 15 as +-448), and every such value (|v| in [2^-5, 448] or 0) is an
// exact fp16. A 16-row slab lies inside one 128-row tile, so the chunk's scales are
// one byte per 128 columns for all of its rows.
template <>
struct Tile<Fp8Rows> {
    static constexpr bool kPermuted = false;
    static constexpr bool kScales = false;
    static constexpr bool kTileScale = true;
    static constexpr uint32_t kChunkGU = 256, kChunkDn = 256;
    static constexpr __host__ __device__ uint32_t wdw(uint32_t kc) { return kc / 4; }  // kc bytes
    static constexpr __host__ __device__ uint32_t sdw(uint32_t) { return 0; }
    static constexpr __host__ __device__ uint32_t lds_dw(uint32_t kc) { return kSlab * (wdw(kc) + 4); }
    static __device__ __forceinline__ size_t wpitch(const Fp8Rows& m) { return m.wrow; }
    static __device__ __forceinline__ size_t spitch(const Fp8Rows&) { return 0; }
    static __device__ __forceinline__ const uint8_t* wrow(const Fp8Rows& m, uint32_t c0) { return m.w + c0; }
    static __device__ __forceinline__ const uint8_t* srow(const Fp8Rows&, uint32_t) { return nullptr; }
    // the scale bytes of the tiles under columns [c0, c0 + kc) (kc <= 512) of row r0's
    // tile row, byte i for columns [c0 + 128 i, c0 + 128 i + 128); c0 % 128 == 0
    static __device__ __forceinline__ uint32_t tile_scales(const Fp8Rows& m, uint32_t r0, uint32_t c0, uint32_t kc) {
        const gptr<uint8_t> s = as_global(m.s + static_cast<size_t>(r0 >> 7) * m.scols + (c0 >> 7));
        const uint32_t n = (kc + 127) >> 7;
        uint32_t v = 0;
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i)
            if (i < n) v |= static_cast<uint32_t>(s[i]) << (8 * i);
        return v;
    }
    static __device__ __forceinline__ half8 get(const uint8_t* w, const uint8_t*, uint32_t ts, uint32_t b, uint32_t kg,
                                                float& scale) {
        scale = e8m0_to_f32((ts >> (8 * (b >> 2))) & 0xFFu);
        const uint32_t d0 = *reinterpret_cast<const uint32_t*>(w + 32 * b + 8 * kg);
        const uint32_t d1 = *reinterpret_cast<const uint32_t*>(w + 32 * b + 8 * kg + 4);
        h2 p[4];  // element order
        fp8x4_to_h2x2(d0, p[0], p[1]);
        fp8x4_to_h2x2(d1, p[2], p[3]);
        return pack8(p[0], p[1], p[2], p[3]);
    }
};

// Buffer loads over one matrix: the per-lane offsets stay in registers of their own
// from chunk to chunk (the chunk's offset is a scalar), so issuing the next chunk's
// loads never waits on registers that earlier loads still write.
// `base` is the same in every lane (a member set's matrix).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t matrix_rsrc(const void* base) {
    const uint64_t a = reinterpret_cast<uint64_t>(base);
    const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(a));
    const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(a >> 32));
    void* p = reinterpret_cast<void*>((static_cast<uint64_t>(hi) << 32) | lo);
    return __builtin_amdgcn_make_buffer_rsrc(p, 0, 0x7FFFFFFF, 0x00020000);
}
}  // namespace dev
}  // namespace objeta

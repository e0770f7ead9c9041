// wide.hip — products of packed matrices with many vectors at once, for prompts and
// large batches: the experts' products for all tokens that selected them and the GEMV
// entry points' large batches.
//
// v_mfma_f32_16x16x32_f16 with the activations as A (16 vectors) and the weights as B
// (16 output rows). Activations come split into two fp16 parts (22 significant bits,
// split_row), weights are exact in fp16, and the row's block scale multiplies the sum of
// a 32-column block in fp32.
//
// Work split: a workgroup takes 128 weight rows (gate/up: 64 of each matrix) and a work
// item of 32 vectors (16 for split FP4), and walks the columns in chunks of 128. Its four
// waves are two row halves times two halves of the chunk's blocks, so one A operand read
// from LDS serves four row tiles and a weight is decoded once per work item. The next
// chunk's loads travel in registers during the products.
//
// What bounds it: latency. At 512 tokens of hidden 2048, intermediate 768, 128 experts,
// top-8 (Q4_0) the matrix cores are about a quarter busy and the VALU (decode, two
// operations per output of a block) a third; three workgroups per CU hide the rest best:
//   64 vectors per work item, two workgroups per CU: 476 us for the layer; 32 vectors,
//   three: 366; 32 vectors in 128 registers (four per CU, 100 bytes of spills): 663.
// The per-assignment kernels took 1893 us for that layer, the eight-member sets of
// grouped.hip 188 us for the 97-token Q5_0 layer that takes 126 here, and eight passes
// of gemv_mfma_kernel 73 us for 64 vectors by 4096 x 4096 (Q4_0; 25.6 here).
//
// Rounding (relative to 64-bit results, against the kernels before): a running sum over
// two chunks, added to a total, keeps the chains short. The two parts' block sums are
// added in fp32: taking both through one MFMA accumulator costs less but the unit
// truncates (5.1e-8 per block instead of 2.6e-8, with the low part first biased by
// 7e-9, which adds up over the blocks). Split FP4 keeps the parts' sums apart (its scales
// are powers of two, so the high parts' sums are nearly exact), which takes the registers
// of a second vector tile. GEMV at 64 vectors 9.4e-8 (before: 1.06e-7), the 512-token
// layer 1.92e-7 (2.13e-7).
#include "mfma_tiles.hpp"

namespace objeta {
namespace {

using namespace dev;

constexpr uint32_t kWMaxTable = 1024;   // experts per table
constexpr uint32_t kWMaxAssign = 4096;  // assignments (tokens * k) per launch
// Vector tiles of 16 per work item (two tiles and the parts' sums apart do not fit 168
// registers: split FP4 at three sums and two tiles spilled 80 to 92 bytes).
template <class R>
constexpr int kWTiles = 2;
template <>
constexpr int kWTiles<Fp4Rows> = 1;
template <class R>
constexpr uint32_t kWMembersOf = 16u * kWTiles<R>;
constexpr uint32_t kWChunk = 128;       // columns per staged chunk
constexpr uint32_t kFlush = 2;          // chunks per running sum
constexpr uint32_t kWRows = 128;        // weight rows per workgroup, over all matrices
constexpr uint32_t kWAStride = kWChunk + 8;  // halves per staged vector part: 68 dwords, so the
                                             // 16 rows of an operand read start 4 banks apart

// One work item: up to 64 assignments that selected the same expert, their act rows
// order[first .. first + count).
struct WideSet {
    objeta_hip_expert_ptrs p;
    uint32_t first, count, pad[2];
};
static_assert(sizeof(WideSet) == 64, "one 64-byte record per set");

struct WideWs {
    uint32_t* hdr;    // [0] number of sets
    WideSet* sets;
    uint2* order;     // {act row, token} grouped by expert, then the shared expert's
};

// Groups the assignments by expert (workgroup of 256). An assignment's place among its
// expert's comes from an LDS atomic, so the order inside an expert is not fixed; it
// decides only which lane multiplies a row, not the row's arithmetic.
__device__ void group_wide(const uint32_t* __restrict__ ids, uint32_t n_assign, uint32_t n_table,
                           const objeta_hip_expert_ptrs* __restrict__ table,
                           const objeta_hip_expert_ptrs* __restrict__ shared, uint32_t n_tokens, WideWs w,
                           uint32_t k, uint32_t members, uint32_t* __restrict__ err) {
    __shared__ uint32_t cnt[kWMaxTable];
    __shared__ uint32_t pos[kWMaxTable];
    __shared__ uint16_t rank[kWMaxAssign];
    __shared__ uint32_t wtot[2][4];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (uint32_t e = tid; e < n_table; e += 256) cnt[e] = 0;
    __syncthreads();
    bool bad = false;
#pragma unroll 4
    for (uint32_t a = tid; a < n_assign; a += 256) {
        const uint32_t e = ids[a];
        if (e < n_table) rank[a] = static_cast<uint16_t>(atomicAdd(&cnt[e], 1u));
        else bad = true;
    }
    if (bad) atomicOr(err, 1u);
    __syncthreads();
    // exclusive prefixes over experts of the counts and of the sets; thread t owns
    // experts [t*per, (t+1)*per)
    const uint32_t per = (n_table + 255) / 256;
    const uint32_t e0 = tid * per < n_table ? tid * per : n_table;
    const uint32_t e1 = e0 + per < n_table ? e0 + per : n_table;
    uint32_t sc = 0, ss = 0;
    for (uint32_t e = e0; e < e1; ++e) {
        sc += cnt[e];
        ss += (cnt[e] + members - 1) / members;
    }
    uint32_t ic = sc, is = ss;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t oc = __shfl_up(ic, off, 64), os = __shfl_up(is, off, 64);
        if (static_cast<int>(lane) >= off) {
            ic += oc;
            is += os;
        }
    }
    if (lane == 63) {
        wtot[0][wave] = ic;
        wtot[1][wave] = is;
    }
    __syncthreads();
    uint32_t bc = 0, bs = 0, tc = 0, ts = 0;
    for (uint32_t v = 0; v < 4; ++v) {
        if (v < wave) {
            bc += wtot[0][v];
            bs += wtot[1][v];
        }
        tc += wtot[0][v];
        ts += wtot[1][v];
    }
    uint32_t pc = bc + ic - sc, ps = bs + is - ss;
    for (uint32_t e = e0; e < e1; ++e) {
        pos[e] = pc;
        for (uint32_t j = 0; j < cnt[e]; j += members) {
            WideSet* dst = &w.sets[ps++];
            dst->p = table[e];
            dst->first = pc + j;
            dst->count = cnt[e] - j < members ? cnt[e] - j : members;
        }
        pc += cnt[e];
    }
    if (shared) {
        const uint32_t n_sh = (n_tokens + members - 1) / members;
        for (uint32_t s = tid; s < n_sh; s += 256) {
            const uint32_t t0 = s * members;
            WideSet* dst = &w.sets[ts + s];
            dst->p = *shared;
            dst->first = tc + t0;
            dst->count = n_tokens - t0 < members ? n_tokens - t0 : members;
        }
        for (uint32_t t = tid; t < n_tokens; t += 256) w.order[tc + t] = make_uint2(n_assign + t, t);
        ts += n_sh;
    }
    if (tid == 0) w.hdr[0] = ts;
    __syncthreads();
#pragma unroll 4
    for (uint32_t a = tid; a < n_assign; a += 256) {
        const uint32_t e = ids[a];
        if (e < n_table) w.order[pos[e] + rank[a]] = make_uint2(a, a / k);
    }
}

// Block 0 groups the assignments; block 1 + t splits row t of x.
__global__ __launch_bounds__(256) void wide_prepare_kernel(const uint32_t* __restrict__ ids, uint32_t n_assign,
                                                           uint32_t n_table,
                                                           const objeta_hip_expert_ptrs* __restrict__ table,
                                                           const objeta_hip_expert_ptrs* __restrict__ shared,
                                                           uint32_t n_tokens, uint32_t k, uint32_t members, WideWs w,
                                                           uint32_t* __restrict__ err,
                                                           const float* __restrict__ x, uint32_t cols,
                                                           _Float16* __restrict__ xh, _Float16* __restrict__ xl,
                                                           float* __restrict__ xmult, uint32_t perm) {
    if (blockIdx.x == 0) group_wide(ids, n_assign, n_table, table, shared, n_tokens, w, k, members, err);
    else split_row(x, cols, xh, xl, xmult, blockIdx.x - 1, perm);
}

// One workgroup per row.
__global__ __launch_bounds__(256) void wide_split_kernel(const float* __restrict__ src, uint32_t cols,
                                                         _Float16* __restrict__ hi, _Float16* __restrict__ lo,
                                                         float* __restrict__ mult, uint32_t perm) {
    split_row(src, cols, hi, lo, mult, blockIdx.x, perm);
}

enum WideMode { kWGateUp = 0, kWDown = 1, kWGemv = 2 };

// LDS of a workgroup: the weight rows (kStride dwords each; an odd multiple of 4, so 16
// rows spread over all banks), the FP4 scale dwords, then both parts of the vectors.
template <class R>
struct WideLds {
    static constexpr uint32_t kSeg = Tile<R>::wdw(kWChunk);  // weight dwords per row and chunk
    static constexpr uint32_t kStride = ((kSeg + 3) / 4 | 1u) * 4;
    static constexpr uint32_t kW = kWRows * kStride;
    static constexpr uint32_t kS = Tile<R>::kScales ? kWRows : 0u;
    static constexpr uint32_t kA = kWMembersOf<R> * kWAStride;  // dwords of both parts
    static constexpr uint32_t kDwords = kW + kS + kA;
};
static_assert(WideLds<QRows<kQ5>>::kStride == 28 && WideLds<QRows<kQ4>>::kStride == 20, "odd multiples of 4");
// the other half's sums (2 row halves x 4 row tiles x 4 vector tiles x 64 lanes x 16 bytes)
static_assert(WideLds<QRows<kIQ3>>::kDwords >= 2 * 4 * kWTiles<QRows<kIQ3>> * 64 * 4, "the sums fit the staging LDS");

// MODE kWGateUp: rows = inter over the split x rows, writes act; kWDown: rows = out_dim
// over the split act rows, writes part; kWGemv: one matrix (w0, s0), vector group
// blockIdx.z, column range blockIdx.y of `range` columns, writes out[range][vec][row].
// The MoE modes take a linear grid: workgroup b runs on XCD b % 8 and takes row block
// (b / 8) % nrb of set b % 8 + 8 * (b / (8 nrb)), so all row blocks of a set read its
// vectors through one L2; sets past the device's count leave at once. FULL: every chunk is whole (else the last has 64 columns).
template <class R, int MODE, bool FULL>
__global__ __launch_bounds__(256, 3) void wide_products_kernel(
    WideWs gw, const void* __restrict__ w0, const void* __restrict__ s0, const _Float16* __restrict__ vh,
    const _Float16* __restrict__ vl, const float* __restrict__ vmult, float* __restrict__ out, uint32_t cols,
    uint32_t rows, uint32_t n_vec, uint32_t range, uint32_t nrb, float limit,
    uint32_t official) {
    constexpr int kMT = kWTiles<R>;
    constexpr uint32_t kWMembers = kWMembersOf<R>;
    using L = WideLds<R>;
    using TR = Tile<R>;
    constexpr int kMats = MODE == kWGateUp ? 2 : 1;
    constexpr bool kApart = TR::kScales;  // the parts' sums apart
    constexpr uint32_t kMatRows = kWRows / kMats;
    constexpr uint32_t kUpr = (L::kSeg + 3) / 4;                // 16-byte units per row
    constexpr uint32_t kNU = (kMatRows * kUpr + 255) / 256;      // units per thread and matrix
    extern __shared__ __align__(16) uint32_t wl[];
    uint32_t* const sl = wl + L::kW;
    _Float16* const al = reinterpret_cast<_Float16*>(wl + L::kW + L::kS);  // [part][member][kWAStride]
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t wr = wave & 1, wk = wave >> 1;
    const uint32_t n16 = lane & 15, kg = lane >> 4;
    __shared__ uint32_t s_row[kWMembers];  // the members' act rows
    __shared__ float s_mul[kWMembers];     // and the powers of two of their split vectors
    uint32_t rb, first, m, c_begin, c_end;
    const void *pw[kMats], *ps[kMats];
    if constexpr (MODE == kWGemv) {
        rb = blockIdx.x;
        c_begin = blockIdx.y * range;
        c_end = c_begin + range < cols ? c_begin + range : cols;
        first = blockIdx.z * kWMembers;
        m = n_vec - first < kWMembers ? n_vec - first : kWMembers;
        pw[0] = w0;
        ps[0] = s0;
    } else {
        const uint32_t b = blockIdx.x, j = b >> 3;
        rb = j % nrb;
        const uint32_t si = (j / nrb) * 8 + (b & 7);
        if (si >= gw.hdr[0]) return;
        c_begin = 0;
        c_end = cols;
        const WideSet& S = gw.sets[si];
        first = S.first;
        m = S.count;
        if constexpr (MODE == kWGateUp) {
            pw[0] = S.p.gate;
            ps[0] = S.p.gate_scale;
            pw[kMats - 1] = S.p.up;
            ps[kMats - 1] = S.p.up_scale;
        } else {
            pw[0] = S.p.down;
            ps[0] = S.p.down_scale;
        }
    }
    const uint32_t r0 = rb * kMatRows;
    const uint32_t nmt = (m + 15) / 16;  // vector tiles
    // {act row, row of the split vectors} of member j (past m: the last)
    auto member = [&](uint32_t j) -> uint2 {
        const uint32_t i = first + (j < m ? j : m - 1);
        if constexpr (MODE == kWGemv) return make_uint2(i, i);
        const uint2 o = gw.order[i];
        return MODE == kWGateUp ? o : make_uint2(o.x, o.x);
    };
    R mt[kMats];
    __amdgpu_buffer_rsrc_t rs[kMats];
#pragma unroll
    for (int t = 0; t < kMats; ++t) {
        mt[t] = RowsOf<R>::make(pw[t], ps[t], cols);
        rs[t] = matrix_rsrc(TR::wrow(mt[t], 0));
    }
    const __amdgpu_buffer_rsrc_t rh = matrix_rsrc(vh), rl = matrix_rsrc(vl);
    const uint32_t wpitch = static_cast<uint32_t>(TR::wpitch(mt[0]));
    // this thread's units: weights (row, dword of the row segment), vectors (8 columns
    // of kMT members)
    uint32_t woff[kNU], wlds[kNU];
    bool wlive[kNU];
#pragma unroll
    for (uint32_t i = 0; i < kNU; ++i) {
        const uint32_t u = threadIdx.x + 256u * i;
        const uint32_t rr = u / kUpr, c = u - rr * kUpr;
        wlive[i] = rr < kMatRows;
        const uint32_t r = r0 + rr < rows ? r0 + rr : rows - 1;
        const uint32_t d = 4 * c < L::kSeg - 4 ? 4 * c : L::kSeg - 4;
        woff[i] = r * wpitch + 4 * d;
        wlds[i] = rr * L::kStride + d;
    }
    const uint32_t ac = threadIdx.x & 15, am = threadIdx.x >> 4;
    uint32_t aoff[kMT];
#pragma unroll
    for (uint32_t i = 0; i < kMT; ++i) aoff[i] = (member(am + 16 * i).y * cols + 8 * ac) * 2;
    u32x4 sw[kMats][kNU], sa[2][kMT];
    uint32_t ssc[kMats] = {}, sts[kMats] = {};
    auto stage = [&](uint32_t c0) {
        const uint32_t kc = FULL || c_end - c0 >= kWChunk ? kWChunk : c_end - c0;
        if (FULL || kc == kWChunk) {
#pragma unroll
            for (int t = 0; t < kMats; ++t) {
                const int so = static_cast<int>(TR::wrow(mt[t], c0) - TR::wrow(mt[t], 0));
#pragma unroll
                for (uint32_t i = 0; i < kNU; ++i)
                    if ((kMatRows * kUpr) % 256 == 0 || wlive[i]) {
                        const auto q = __builtin_amdgcn_raw_buffer_load_b128(rs[t], static_cast<int>(woff[i]), so, 0);
                        sw[t][i] = u32x4{q[0], q[1], q[2], q[3]};
                    }
            }
#pragma unroll
            for (uint32_t i = 0; i < kMT; ++i)
                if (i < nmt) {
                    const auto q = __builtin_amdgcn_raw_buffer_load_b128(rh, static_cast<int>(aoff[i]), static_cast<int>(2 * c0), 0);
                    sa[0][i] = u32x4{q[0], q[1], q[2], q[3]};
                    const auto p = __builtin_amdgcn_raw_buffer_load_b128(rl, static_cast<int>(aoff[i]), static_cast<int>(2 * c0), 0);
                    sa[1][i] = u32x4{p[0], p[1], p[2], p[3]};
                }
        } else {  // a last chunk of 64 columns: half the units, shifted inside the row
            const uint32_t seg = TR::wdw(kc);
#pragma unroll
            for (int t = 0; t < kMats; ++t) {
                const int so = static_cast<int>(TR::wrow(mt[t], c0) - TR::wrow(mt[t], 0));
#pragma unroll
                for (uint32_t i = 0; i < kNU; ++i) {
                    const uint32_t u = threadIdx.x + 256u * i;
                    const uint32_t rr = u / kUpr, c = u - rr * kUpr;
                    if (rr < kMatRows && 4 * c < seg) {
                        const uint32_t r = r0 + rr < rows ? r0 + rr : rows - 1;
                        const uint32_t d = 4 * c < seg - 4 ? 4 * c : seg - 4;
                        const auto q = __builtin_amdgcn_raw_buffer_load_b128(rs[t], static_cast<int>(r * wpitch + 4 * d), so, 0);
                        sw[t][i] = u32x4{q[0], q[1], q[2], q[3]};
                    }
                }
            }
#pragma unroll
            for (uint32_t i = 0; i < kMT; ++i)
                if (i < nmt && 8 * ac < kc) {
                    const auto q = __builtin_amdgcn_raw_buffer_load_b128(rh, static_cast<int>(aoff[i]), static_cast<int>(2 * c0), 0);
                    sa[0][i] = u32x4{q[0], q[1], q[2], q[3]};
                    const auto p = __builtin_amdgcn_raw_buffer_load_b128(rl, static_cast<int>(aoff[i]), static_cast<int>(2 * c0), 0);
                    sa[1][i] = u32x4{p[0], p[1], p[2], p[3]};
                }
        }
        if constexpr (TR::kScales) {  // one dword of E8M0 bytes per row
#pragma unroll
            for (int t = 0; t < kMats; ++t)
                if (threadIdx.x < kMatRows) {
                    const uint32_t r = r0 + threadIdx.x < rows ? r0 + threadIdx.x : rows - 1;
                    ssc[t] = *as_global(reinterpret_cast<const uint32_t*>(TR::srow(mt[t], c0) +
                                                                          static_cast<size_t>(r) * TR::spitch(mt[t])));
                }
        }
        if constexpr (TR::kTileScale)
#pragma unroll
            for (int t = 0; t < kMats; ++t) sts[t] = TR::tile_scales(mt[t], r0, c0, kWChunk);
    };
    uint32_t ts_cur[kMats] = {};
    auto commit = [&](uint32_t c0) {
        const uint32_t kc = FULL || c_end - c0 >= kWChunk ? kWChunk : c_end - c0;
        typedef uint32_t u32x2s __attribute__((ext_vector_type(2), aligned(8)));
        typedef uint32_t u32x4s __attribute__((ext_vector_type(4), aligned(16)));
#pragma unroll
        for (int t = 0; t < kMats; ++t) {
            uint32_t* base = wl + t * kMatRows * L::kStride;
            if (FULL || kc == kWChunk) {
#pragma unroll
                for (uint32_t i = 0; i < kNU; ++i)
                    if ((kMatRows * kUpr) % 256 == 0 || wlive[i]) {
                        *reinterpret_cast<u32x2s*>(base + wlds[i]) = u32x2s{sw[t][i].x, sw[t][i].y};
                        *reinterpret_cast<u32x2s*>(base + wlds[i] + 2) = u32x2s{sw[t][i].z, sw[t][i].w};
                    }
            } else {
                const uint32_t seg = TR::wdw(kc);
#pragma unroll
                for (uint32_t i = 0; i < kNU; ++i) {
                    const uint32_t u = threadIdx.x + 256u * i;
                    const uint32_t rr = u / kUpr, c = u - rr * kUpr;
                    if (rr < kMatRows && 4 * c < seg) {
                        const uint32_t d = 4 * c < seg - 4 ? 4 * c : seg - 4;
                        uint32_t* dst = base + rr * L::kStride + d;
                        dst[0] = sw[t][i].x; dst[1] = sw[t][i].y; dst[2] = sw[t][i].z; dst[3] = sw[t][i].w;
                    }
                }
            }
            if constexpr (TR::kScales)
                if (threadIdx.x < kMatRows) sl[t * kMatRows + threadIdx.x] = ssc[t];
            ts_cur[t] = sts[t];
        }
#pragma unroll
        for (uint32_t i = 0; i < kMT; ++i)
            if (i < nmt && (FULL || 8 * ac < kc)) {
                _Float16* dst = al + (am + 16 * i) * kWAStride + 8 * ac;
                *reinterpret_cast<u32x4s*>(dst) = u32x4s{sa[0][i].x, sa[0][i].y, sa[0][i].z, sa[0][i].w};
                *reinterpret_cast<u32x4s*>(dst + kWMembers * kWAStride) =
                    u32x4s{sa[1][i].x, sa[1][i].y, sa[1][i].z, sa[1][i].w};
            }
    };
    // [row tile][vector tile]: the running sums of up to kFlush chunks, and of those
    f32x4 acc[4][kMT], accl[4][kMT], total[4][kMT];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < kMT; ++b) acc[a][b] = accl[a][b] = total[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    // LDS row of this lane in row tile rt, and that tile's matrix
    auto tile_mat = [&](int rt) { return MODE == kWGateUp ? rt >> 1 : 0; };
    auto tile_row = [&](int rt) {
        return MODE == kWGateUp ? wr * 32u + static_cast<uint32_t>(rt & 1) * 16u + n16
                                : wr * 64u + static_cast<uint32_t>(rt) * 16u + n16;
    };
    // the products of block b of the chunk with vector tiles 0 .. MT - 1
    auto block = [&](uint32_t b, auto mtc) {
        constexpr int MT = decltype(mtc)::value;
        half8 xh[MT], xl[MT];
#pragma unroll
        for (int v = 0; v < MT; ++v) {
            const _Float16* src = al + (16u * v + n16) * kWAStride + 32u * b + 8u * kg;
            xh[v] = *reinterpret_cast<const half8*>(src);
            xl[v] = *reinterpret_cast<const half8*>(src + kWMembers * kWAStride);
        }
#pragma unroll
        for (int rt = 0; rt < 4; ++rt) {
            const uint32_t lr = tile_mat(rt) * kMatRows + tile_row(rt);
            float sc;
            const half8 bw = TR::get(reinterpret_cast<const uint8_t*>(wl + lr * L::kStride),
                                     reinterpret_cast<const uint8_t*>(sl + lr), ts_cur[tile_mat(rt)], b, kg, sc);
            f32x4 zh[MT], zl[MT];
            const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int v = 0; v < MT; ++v) zh[v] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh[v], bw, zero, 0, 0, 0);
#pragma unroll
            for (int v = 0; v < MT; ++v) zl[v] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xl[v], bw, zero, 0, 0, 0);
#pragma unroll
            for (int v = 0; v < MT; ++v)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    if constexpr (kApart) {
                        acc[rt][v][q] = __builtin_fmaf(sc, zh[v][q], acc[rt][v][q]);
                        accl[rt][v][q] = __builtin_fmaf(sc, zl[v][q], accl[rt][v][q]);
                    } else {
                        acc[rt][v][q] = __builtin_fmaf(sc, zh[v][q] + zl[v][q], acc[rt][v][q]);
                    }
                }
        }
    };
    uint32_t pending = 0;  // chunks in acc
    stage(c_begin);
    for (uint32_t c0 = c_begin; c0 < c_end; c0 += kWChunk) {
        const uint32_t kc = FULL || c_end - c0 >= kWChunk ? kWChunk : c_end - c0;
        __syncthreads();  // the previous chunk's (or set's) LDS reads are done
        commit(c0);
        __syncthreads();
        if (c0 + kWChunk < c_end) stage(c0 + kWChunk);  // in flight during the products
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        const uint32_t per = FULL ? 2u : kc / 64;  // blocks of this wave's half
#pragma unroll 1
        for (uint32_t i = 0; i < per; ++i) {
            const uint32_t b = wk * per + i;
            if (kMT == 1 || nmt > 1) block(b, std::integral_constant<int, kMT>{});
            else block(b, std::integral_constant<int, 1>{});
        }
        if (++pending == (kApart ? 4 : kFlush)) {
            pending = 0;
#pragma unroll
            for (int a = 0; a < 4; ++a)
#pragma unroll
                for (int v = 0; v < kMT; ++v) {
                    if constexpr (kApart) acc[a][v] += accl[a][v];
                    total[a][v] += acc[a][v];
                    acc[a][v] = accl[a][v] = f32x4{0.f, 0.f, 0.f, 0.f};
                }
        }
    }
    if (threadIdx.x < kWMembers) {
        const uint2 o = member(threadIdx.x);
        s_row[threadIdx.x] = o.x;
        s_mul[threadIdx.x] = vmult[o.y];
    }
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int v = 0; v < kMT; ++v) {
            if constexpr (kApart) acc[a][v] += accl[a][v];
            total[a][v] += acc[a][v];
        }
    // the two column halves meet in LDS: wave (wr, wk) finishes vector tiles v with
    // v % 2 == wk and hands the others over
    f32x4* const red = reinterpret_cast<f32x4*>(wl) + wr * 4 * kMT * 64;
    __syncthreads();
#pragma unroll
    for (int v = 0; v < kMT; ++v)
        if ((v & 1) != static_cast<int>(wk) && static_cast<uint32_t>(v) < nmt) {
#pragma unroll
            for (int rt = 0; rt < 4; ++rt) red[(v * 4 + rt) * 64 + lane] = total[rt][v];
        }
    __syncthreads();
    // lane: weight row n16 of the tile, members 16 v + 4 kg + q
#pragma unroll
    for (int v = 0; v < kMT; ++v) {
        if ((v & 1) != static_cast<int>(wk) || static_cast<uint32_t>(v) >= nmt) continue;
#pragma unroll
        for (int rt = 0; rt < 4; ++rt) total[rt][v] += red[(v * 4 + rt) * 64 + lane];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint32_t j = 16u * v + 4u * kg + static_cast<uint32_t>(q);
            const float mul = s_mul[j];
            const size_t at = MODE == kWGemv ? (static_cast<size_t>(blockIdx.y) * n_vec + s_row[j]) * rows
                                             : static_cast<size_t>(s_row[j]) * rows;
            if constexpr (MODE == kWGateUp) {
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const uint32_t r = r0 + tile_row(h);
                    if (j < m && r < rows)
                        out[at + r] = swiglu(total[h][v][q] * mul, total[h + 2][v][q] * mul, limit, official);
                }
            } else {
#pragma unroll
                for (int rt = 0; rt < 4; ++rt) {
                    const uint32_t r = r0 + tile_row(rt);
                    if (j < m && r < rows) out[at + r] = total[rt][v][q] * mul;
                }
            }
        }
    }
}

size_t al256(size_t v) { return (v + 255) & ~size_t(255); }

template <class R, int MODE>
void launch_wide_products(hipStream_t s, dim3 grid, WideWs gw, const void* w0, const void* s0, const _Float16* vh,
                          const _Float16* vl, const float* vmult, float* dst, uint32_t cols, uint32_t rows,
                          uint32_t n_vec, uint32_t range, uint32_t nrb, float limit, bool official) {
    const size_t lds = 4 * static_cast<size_t>(WideLds<R>::kDwords);
    if (Tile<R>::kScales || cols % kWChunk == 0)  // split FP4 rows are whole chunks
        hipLaunchKernelGGL((wide_products_kernel<R, MODE, true>), grid, dim3(256), lds, s, gw, w0, s0, vh, vl, vmult, dst,
                           cols, rows, n_vec, range, nrb, limit, official ? 1u : 0u);
    else if constexpr (!Tile<R>::kScales)
        hipLaunchKernelGGL((wide_products_kernel<R, MODE, false>), grid, dim3(256), lds, s, gw, w0, s0, vh, vl, vmult, dst,
                           cols, rows, n_vec, range, nrb, limit, official ? 1u : 0u);
}

// One phase of the grouped experts: as many workgroups as there can be (row block,
// set) pairs; a set's number is below max_sets, the real count is known on the device.
template <class R, int MODE>
void launch_wide_phase(hipStream_t s, WideWs gw, const _Float16* vh, const _Float16* vl, const float* vmult, float* dst,
                       uint32_t cols, uint32_t rows, uint32_t max_sets, float limit,
                       bool official) {
    const uint32_t mr = MODE == kWGateUp ? kWRows / 2 : kWRows;
    const uint32_t nrb = (rows + mr - 1) / mr;
    launch_wide_products<R, MODE>(s, dim3(8 * nrb * ((max_sets + 7) / 8)), gw, nullptr, nullptr, vh, vl, vmult, dst, cols,
                                  rows, 0, 0, nrb, limit, official);
}

template <class R>
void launch_wide_layer(hipStream_t s, WideWs gw, const _Float16* xh, const _Float16* xl, const float* xmult, float* act,
                       _Float16* ah, _Float16* al, float* amult, float* part, uint32_t n_rows,
                       uint32_t max_sets, uint32_t hidden, uint32_t inter, uint32_t out_dim, float limit) {
    launch_wide_phase<R, kWGateUp>(s, gw, xh, xl, xmult, act, hidden, inter, max_sets, limit, false);
    hipLaunchKernelGGL(wide_split_kernel, dim3(n_rows), dim3(256), 0, s, act, inter, ah, al, amult,
                       Tile<R>::kPermuted ? 1u : 0u);
    launch_wide_phase<R, kWDown>(s, gw, ah, al, amult, part, inter, out_dim, max_sets, 0.0f, false);
}

// Offsets in the kernels are 32-bit: matrices and split vectors below 2^31 bytes.
bool below_2g(uint64_t rows, uint64_t bytes_per_row) { return rows * bytes_per_row < (uint64_t(1) << 31); }

}  // namespace

bool wide_supported(int32_t format, uint64_t n_table, uint64_t n_tokens, uint64_t k, uint64_t hidden, uint64_t inter,
                    uint64_t out_dim) {
    if (format < OBJETA_HIP_Q4_0 || format > OBJETA_HIP_FP4_E2M1) return false;
    if (k == 0 || k > 32 || n_table == 0 || n_table > kWMaxTable || n_tokens < kWideMinTokens || out_dim == 0) return false;
    if (hidden == 0 || inter == 0 || hidden % 64 || inter % 64 || hidden > (1u << 20) || inter > (1u << 20) ||
        out_dim > (1u << 20))
        return false;
    if (format == OBJETA_HIP_FP4_E2M1 && (hidden % 128 || inter % 128)) return false;
    const uint64_t t = n_tokens < kWMaxAssign / k ? n_tokens : kWMaxAssign / k;  // tokens of a launch
    return below_2g(inter, hidden) && below_2g(out_dim, inter) && below_2g(t, 2 * hidden) &&
           below_2g(t * (k + 1), 2 * inter);
}

int32_t launch_moe_wide(objeta_hip_context* ctx, int32_t format, hipStream_t s, const objeta_hip_expert_ptrs* table,
                        uint64_t n_table, const objeta_hip_expert_ptrs* shared, const uint32_t* ids, const float* wts,
                        uint64_t n_tokens, uint64_t k, const float* x, const float* resid, float* out, uint64_t hidden,
                        uint64_t inter, uint64_t out_dim, float limit) {
    const char* action = "launch grouped-token MoE (wide)";
    if (!wide_supported(format, n_table, n_tokens, k, hidden, inter, out_dim))
        OBJ_FAIL(kUnsupported, action, "shape outside the wide products");
    if (!table || !ids || !wts || !x || !out) OBJ_FAIL(kInvalidInput, action, "NULL device pointer");
    if (reinterpret_cast<uintptr_t>(x) % 16) OBJ_FAIL(kInvalidInput, action, "x must be 16-byte aligned");
    const uint32_t H = static_cast<uint32_t>(hidden), I = static_cast<uint32_t>(inter), O = static_cast<uint32_t>(out_dim);
    const uint32_t M = format == OBJETA_HIP_FP4_E2M1 ? kWMembersOf<Fp4Rows> : kWMembersOf<QRows<kQ4>>;
    const uint32_t kk = static_cast<uint32_t>(k), E = static_cast<uint32_t>(n_table);
    // tokens in equal slices of at most kWMaxAssign assignments (the workspace of a
    // slice is reused by the next)
    const uint64_t per = kWMaxAssign / k, slices = (n_tokens + per - 1) / per;
    const uint64_t slice = (n_tokens + slices - 1) / slices;
    const uint32_t T = static_cast<uint32_t>(slice), A = T * kk;
    const uint32_t NR = A + (shared ? T : 0);  // act rows: routed, then shared
    const uint32_t NS = (A < E ? A : E) + A / M + (shared ? (T + M - 1) / M : 0);
    size_t off = 0;
    const size_t o_hdr = off; off += al256(16);
    const size_t o_set = off; off += al256(sizeof(WideSet) * NS);
    const size_t o_ord = off; off += al256(8ull * NR);
    const size_t o_xm = off; off += al256(4ull * T);
    const size_t o_am = off; off += al256(4ull * NR);
    const size_t o_xh = off; off += al256(2ull * T * H);
    const size_t o_xl = off; off += al256(2ull * T * H);
    const size_t o_act = off; off += al256(4ull * NR * I);
    const size_t o_ah = off; off += al256(2ull * NR * I);
    const size_t o_all = off; off += al256(2ull * NR * I);
    const size_t o_part = off; off += al256(4ull * NR * O);
    void* wsp = nullptr;
    OBJ_TRY(ensure_workspace(ctx, s, kWsGrouped, off, &wsp));
    char* b = static_cast<char*>(wsp);
    const WideWs gw{reinterpret_cast<uint32_t*>(b + o_hdr), reinterpret_cast<WideSet*>(b + o_set),
                    reinterpret_cast<uint2*>(b + o_ord)};
    float* xmult = reinterpret_cast<float*>(b + o_xm);
    float* amult = reinterpret_cast<float*>(b + o_am);
    auto* xh = reinterpret_cast<_Float16*>(b + o_xh);
    auto* xl = reinterpret_cast<_Float16*>(b + o_xl);
    float* act = reinterpret_cast<float*>(b + o_act);
    auto* ah = reinterpret_cast<_Float16*>(b + o_ah);
    auto* all = reinterpret_cast<_Float16*>(b + o_all);
    float* part = reinterpret_cast<float*>(b + o_part);
    const bool perm = format == OBJETA_HIP_FP4_E2M1 ? Tile<Fp4Rows>::kPermuted : Tile<QRows<kQ4>>::kPermuted;
    for (uint64_t t0 = 0; t0 < n_tokens; t0 += slice) {
        const uint32_t t = static_cast<uint32_t>(n_tokens - t0 < slice ? n_tokens - t0 : slice), a = t * kk;
        const uint32_t nr = a + (shared ? t : 0);
        const uint32_t ns = (a < E ? a : E) + a / M + (shared ? (t + M - 1) / M : 0);
        const uint32_t* idt = ids + t0 * k;
        hipLaunchKernelGGL(wide_prepare_kernel, dim3(1 + t), dim3(256), 0, s, idt, a, E, table, shared, t, kk, M, gw,
                           ctx->err_word, x + t0 * hidden, H, xh, xl, xmult, perm ? 1u : 0u);
#define OBJ_WIDE(R) \
    launch_wide_layer<R>(s, gw, xh, xl, xmult, act, ah, all, amult, part, nr, ns, H, I, O, limit)
        switch (format) {
            case OBJETA_HIP_Q4_0: OBJ_WIDE(QRows<kQ4>); break;
            case OBJETA_HIP_Q5_0: OBJ_WIDE(QRows<kQ5>); break;
            case OBJETA_HIP_IQ3_0: OBJ_WIDE(QRows<kIQ3>); break;
            default: OBJ_WIDE(Fp4Rows); break;
        }
#undef OBJ_WIDE
        launch_moe_combine(s, idt, wts + t0 * k, part, shared ? part + static_cast<size_t>(a) * O : nullptr,
                           resid ? resid + t0 * out_dim : nullptr, out + t0 * out_dim, t, kk, O, E);
        OBJ_HIP(hipGetLastError(), action);
    }
    return 0;
}

bool gemv_wide_supported(int32_t format, uint64_t rows, uint64_t cols, uint64_t batch) {
    return batch >= kGemvWideMinBatch && below_2g(rows, cols) && below_2g(batch, 2 * cols) && (batch + 15) / 16 <= 65535;
}

int32_t launch_gemv_wide(objeta_hip_context* ctx, hipStream_t s, int32_t format, const void* w, const void* ws,
                         const float* x, float* y, uint64_t rows, uint64_t cols, uint64_t batch) {
    const char* action = "launch batched GEMV (wide)";
    const uint32_t R = static_cast<uint32_t>(rows), K = static_cast<uint32_t>(cols), B = static_cast<uint32_t>(batch);
    const uint32_t cus = ctx->info.compute_units > 0 ? static_cast<uint32_t>(ctx->info.compute_units) : 256u;
    const uint32_t M = format == OBJETA_HIP_FP4_E2M1 ? kWMembersOf<Fp4Rows> : kWMembersOf<QRows<kQ4>>;
    const uint32_t nrb = (R + kWRows - 1) / kWRows, ng = (B + M - 1) / M;
    // column ranges for about two workgroups per CU, of at least four chunks
    const uint32_t chunks = (K + kWChunk - 1) / kWChunk;
    uint32_t ks = (2 * cus + nrb * ng - 1) / (nrb * ng);
    if (ks > (chunks + 3) / 4) ks = (chunks + 3) / 4;
    const uint32_t rc = (chunks + ks - 1) / ks;  // chunks per range
    ks = (chunks + rc - 1) / rc;
    size_t off = 0;
    const size_t o_xm = off; off += al256(4ull * B);
    const size_t o_xh = off; off += al256(2ull * B * K);
    const size_t o_xl = off; off += al256(2ull * B * K);
    const size_t o_part = off; off += ks > 1 ? al256(4ull * ks * B * R) : 0;
    void* wsp = nullptr;
    OBJ_TRY(ensure_workspace(ctx, s, kWsGemv, off, &wsp));
    char* b = static_cast<char*>(wsp);
    float* xmult = reinterpret_cast<float*>(b + o_xm);
    auto* xh = reinterpret_cast<_Float16*>(b + o_xh);
    auto* xl = reinterpret_cast<_Float16*>(b + o_xl);
    float* part = ks > 1 ? reinterpret_cast<float*>(b + o_part) : y;
    const bool perm = format == OBJETA_HIP_FP4_E2M1 ? Tile<Fp4Rows>::kPermuted : Tile<QRows<kQ4>>::kPermuted;
    hipLaunchKernelGGL(wide_split_kernel, dim3(B), dim3(256), 0, s, x, K, xh, xl, xmult, perm ? 1u : 0u);
    const dim3 grid(nrb, ks, ng);
#define OBJ_WIDE(RT)                                                                                                  \
    launch_wide_products<RT, kWGemv>(s, grid, WideWs{}, w, ws, xh, xl, xmult, part, K, R, B, rc * kWChunk, nrb, 0.0f, \
                                     false)
    switch (format) {
        case OBJETA_HIP_Q4_0: OBJ_WIDE(QRows<kQ4>); break;
        case OBJETA_HIP_Q5_0: OBJ_WIDE(QRows<kQ5>); break;
        case OBJETA_HIP_IQ3_0: OBJ_WIDE(QRows<kIQ3>); break;
        default: OBJ_WIDE(Fp4Rows); break;
    }
#undef OBJ_WIDE
    if (ks > 1) launch_gemv_reduce(s, part, y, R, B, ks);
    OBJ_HIP(hipGetLastError(), action);
    return 0;
}

}  // namespace objeta

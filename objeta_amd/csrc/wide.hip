// wide.hip — products of packed matrices with many vectors at once, for prompts and
// large batches: the experts' products for all tokens that selected them and the GEMV
// entry points' large batches.
//
// v_mfma_f32_16x16x32_f16 with the activations as A (16 vectors) and the weights as B
// (16 output rows). Activations come split into two fp16 parts (22 significant bits,
// split_row), weights are exact in fp16, and the row's block scale multiplies the sum of
// a 32-column block in fp32.
//
// Work split: a workgroup takes 64 or 128 weight rows (gate/up: half of each matrix) and
// a work item of 16 or 32 vectors, and walks the columns in chunks (Work, below). Its four
// waves are two row halves times two halves of the chunk's blocks, so one A operand read
// from LDS serves all row tiles of a wave and a weight is decoded once per work item. The
// next chunk's loads travel in registers during the products.
//
// What bounds it: with few vectors per expert the weights' loads in flight (3.1 to 3.4
// TB/s); with many, latency and the LDS reads. At 512 tokens of hidden 2048, intermediate
// 768, 128 experts, top-8 (Q4_0) the matrix cores are about a quarter busy and the VALU a
// third. Layer times there by shape (vectors, rows, columns of a chunk; workgroups per CU),
// all on one input whose router selection alone takes 78 us:
// 64, 128, 128; 2: 476 us. 32, 128, 128; 3: 353 (in 128 registers, 100 bytes of spills: 663).
// 32, 64, 256; 4: 440. 32, 64, 128; 5: 570. 32, 256, 128; 2: 419. 32, 128, 256; 2: 388. 16, 64,
// 256; 4: 376. Over inputs in turn, before and now: that layer 1844 -> 311 us (the
// per-assignment kernels), a 97-token Q5_0 layer 195 -> 133 (sets of eight), 64 vectors by
// 4096 x 4096 (Q4_0) 74 -> 25 (eight passes of gemv_mfma_kernel).
//
// Rounding (relative to 64-bit results, against the kernels before): a running sum over
// 256 columns (split FP4: 512), added to a total, keeps the chains short. The two parts'
// block sums are added in fp32: taking both through one MFMA accumulator costs less but the
// unit truncates (5.1e-8 per block instead of 2.6e-8, with the low part first biased by
// 7e-9, which adds up over the blocks). Split FP4 keeps the parts' sums apart (its scales
// are powers of two, so the high parts' sums are nearly exact). GEMV at 64 vectors 9.4e-8
// (before: 1.06e-7), the 512-token layer 1.92e-7 (2.13e-7).
#include "mfma_tiles.hpp"

namespace objeta {
namespace {

using namespace dev;

constexpr uint32_t kWMaxTable = 1024;   // experts per table
constexpr uint32_t kWMaxAssign = 4096;  // assignments (tokens * k) per launch

// The shape of a workgroup's work: MT vector tiles of 16 per work item, RT row tiles of
// 16 per wave (32 RT weight rows per workgroup, over all matrices), CH columns per staged
// chunk, W waves per SIMD, the parts of the vectors (1: the low parts are zero).
template <int MT, int RT, uint32_t CH, int W, int PARTS = 2>
struct Work {
    static constexpr int kMT = MT, kRT = RT, kWaves = W, kParts = PARTS;
    static constexpr uint32_t kMembers = 16 * MT, kRows = 32 * RT, kChunk = CH;
};
// Large matrices at many vectors; small ones or few vectors (more workgroups, longer
// chunks); large split FP4 ones (whose sums of the two parts stay apart, which takes the
// registers of a second vector tile: three sums and two tiles spilled 80 to 92 bytes);
// the official layer's, whose vectors have no low part.
using WorkLarge = Work<2, 4, 128, 3>;
using WorkSmall = Work<1, 2, 256, 4>;
using WorkLarge4 = Work<1, 4, 256, 4>;
using WorkOfficial = Work<1, 4, 256, 4, 1>;
using WorkOfficialSmall = Work<1, 2, 256, 4, 1>;

// One work item: assignments that selected the same expert, its table entry copied in and
// their act rows (past count: the last one), so a workgroup reaches its weights and
// vectors through one load.
struct WideSet {
    objeta_hip_expert_ptrs p;
    uint32_t count, pad[3];
    uint16_t row[32];
};
static_assert(sizeof(WideSet) == kWideSetBytes, "one line per set");

// Groups the assignments by expert (workgroup of 256). An assignment's place among its
// expert's comes from an LDS atomic, so the order inside an expert is not fixed; it
// decides only which lane multiplies a row, not the row's arithmetic.
// The shared expert (when given) follows as one more group of `shared_members` per set:
// member t is token t, its act row n_assign + t; its sets go to shared_sets, their number
// to hdr[1] (hdr[0]: the routed sets), or after the routed ones when shared_sets is NULL.
__device__ void group_wide(const uint32_t* __restrict__ ids, uint32_t n_assign, uint32_t n_table,
                           const objeta_hip_expert_ptrs* __restrict__ table,
                           const objeta_hip_expert_ptrs* __restrict__ shared, uint32_t n_tokens, uint32_t members,
                           uint32_t* __restrict__ hdr, WideSet* __restrict__ sets, WideSet* __restrict__ shared_sets,
                           uint32_t* __restrict__ err) {
    __shared__ uint32_t cnt[kWMaxTable];
    __shared__ uint16_t first[kWMaxTable];  // the expert's first set
    __shared__ uint16_t rank[kWMaxAssign];
    __shared__ uint32_t wtot[4];
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
    // exclusive prefix over experts of the sets; thread t owns experts [t*per, (t+1)*per)
    const uint32_t per = (n_table + 255) / 256;
    const uint32_t e0 = tid * per < n_table ? tid * per : n_table;
    const uint32_t e1 = e0 + per < n_table ? e0 + per : n_table;
    uint32_t ss = 0;
    for (uint32_t e = e0; e < e1; ++e) ss += (cnt[e] + members - 1) / members;
    uint32_t is = ss;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t os = __shfl_up(is, off, 64);
        if (static_cast<int>(lane) >= off) is += os;
    }
    if (lane == 63) wtot[wave] = is;
    __syncthreads();
    uint32_t ps = is - ss, ts = 0;
    for (uint32_t v = 0; v < 4; ++v) {
        if (v < wave) ps += wtot[v];
        ts += wtot[v];
    }
    for (uint32_t e = e0; e < e1; ++e) {
        first[e] = static_cast<uint16_t>(ps);
        for (uint32_t j = 0; j < cnt[e]; j += members) {
            WideSet* dst = &sets[ps++];
            dst->p = table[e];
            dst->count = cnt[e] - j < members ? cnt[e] - j : members;
        }
    }
    const uint32_t n_sh = shared ? (n_tokens + members - 1) / members : 0;
    WideSet* const sh = shared_sets ? shared_sets : sets + ts;
    for (uint32_t i = tid; i < n_sh * members; i += 256) {
        const uint32_t t = i < n_tokens ? i : n_tokens - 1;
        WideSet* dst = &sh[i / members];
        dst->row[i % members] = static_cast<uint16_t>(n_assign + t);
        if (i % members == 0) {
            dst->p = *shared;
            dst->count = n_tokens - i < members ? n_tokens - i : members;
        }
    }
    if (tid == 0) {
        hdr[0] = shared_sets ? ts : ts + n_sh;
        hdr[1] = n_sh;
    }
    __syncthreads();
#pragma unroll 4
    for (uint32_t a = tid; a < n_assign; a += 256) {
        const uint32_t e = ids[a];
        if (e >= n_table) continue;
        const uint32_t r = rank[a];
        WideSet* dst = &sets[first[e] + r / members];
        dst->row[r % members] = static_cast<uint16_t>(a);
        if (r + 1 == cnt[e])  // the last one fills the rest of its set
            for (uint32_t q = r % members + 1; q < members; ++q) dst->row[q] = static_cast<uint16_t>(a);
    }
}

// Block 0 groups the assignments; block 1 + t splits row t of x.
__global__ __launch_bounds__(256) void wide_prepare_kernel(
    const uint32_t* __restrict__ ids, uint32_t n_assign, uint32_t n_table,
    const objeta_hip_expert_ptrs* __restrict__ table, const objeta_hip_expert_ptrs* __restrict__ shared,
    uint32_t n_tokens, uint32_t members, uint32_t* __restrict__ hdr, WideSet* __restrict__ sets,
    WideSet* __restrict__ shared_sets, uint32_t* __restrict__ err, const float* __restrict__ x, uint32_t cols,
    _Float16* __restrict__ xh, _Float16* __restrict__ xl, float* __restrict__ xmult, uint32_t perm) {
    if (blockIdx.x == 0)
        group_wide(ids, n_assign, n_table, table, shared, n_tokens, members, hdr, sets, shared_sets, err);
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
// rows spread over all banks), the FP4 scale dwords, then both parts of the vectors
// (rows padded by 8 halves: 4 dwords past a multiple of 64, so the 16 rows of an operand
// read start 4 banks apart).
template <class R, class K>
struct WideLds {
    static constexpr uint32_t kSeg = Tile<R>::wdw(K::kChunk);  // weight dwords per row and chunk
    static constexpr uint32_t kStride = ((kSeg + 3) / 4 | 1u) * 4;
    static constexpr uint32_t kSdw = Tile<R>::kScales ? Tile<R>::sdw(K::kChunk) : 0u;
    static constexpr uint32_t kAStride = K::kChunk + 8;  // halves per staged vector part
    static constexpr uint32_t kW = K::kRows * kStride;
    static constexpr uint32_t kS = K::kRows * kSdw;
    static constexpr uint32_t kA = K::kMembers * kAStride * K::kParts / 2;  // dwords
    static constexpr uint32_t kDwords = kW + kS + kA;
    // the other column half's sums: 2 row halves x RT x MT tiles x 64 lanes x 16 bytes
    static_assert(kDwords >= 2u * K::kRT * K::kMT * 64 * 4, "the sums fit the staging LDS");
};

// MODE kWGateUp: rows = inter over the split x rows, writes act; kWDown: rows = out_dim
// over the split act rows, writes part; kWGemv: one matrix (w0, s0), vector group
// blockIdx.z, column range blockIdx.y of `range` columns, writes out[range][vec][row].
// The MoE modes take a linear grid: workgroup b runs on XCD b % 8 and takes row block
// (b / 8) % nrb of set b % 8 + 8 * (b / (8 nrb)), so all row blocks of a set read its
// vectors through one L2; sets past the device's count leave at once. FULL: every chunk is whole.
struct WideArgs {
    const uint32_t* n;     // number of sets (MoE modes)
    const WideSet* sets;
    const void *w0, *s0;   // the matrix (kWGemv)
    const _Float16 *vh, *vl;
    const float* vmult;
    float* out;
    uint32_t cols, rows, k_inv, n_assign, n_vec, range, nrb;
    float limit;
    uint32_t official;
};

template <class R, class K, int MODE, bool FULL>
__device__ __forceinline__ void wide_body(const WideArgs& g, const uint32_t* __restrict__ set_count,
                                          const WideSet* __restrict__ sets, uint32_t wg) {
    using L = WideLds<R, K>;
    using TR = Tile<R>;
    constexpr int kMT = K::kMT, kRT = K::kRT, kParts = K::kParts;
    constexpr uint32_t kMembers = K::kMembers, kChunk = K::kChunk;
    constexpr int kMats = MODE == kWGateUp ? 2 : 1;
    constexpr bool kApart = TR::kScales && kParts == 2;  // the parts' sums apart
    constexpr uint32_t kFlush = (TR::kScales || kParts == 1 ? 8 : 4) * 64 / kChunk;  // chunks per running sum
    constexpr uint32_t kMatRows = K::kRows / kMats;
    constexpr uint32_t kUpr = (L::kSeg + 3) / 4;                // 16-byte units per row
    constexpr uint32_t kNU = (kMatRows * kUpr + 255) / 256;      // units per thread and matrix
    constexpr uint32_t kAUpr = kChunk / 8;                       // 16-byte units of a vector part
    constexpr uint32_t kAStep = 256 / kAUpr;                     // vectors per round of units
    constexpr uint32_t kNA = kMembers / kAStep;                  // rounds
    const uint32_t cols = g.cols, rows = g.rows, n_assign = g.n_assign, n_vec = g.n_vec, nrb = g.nrb;
    const _Float16* __restrict__ const vh = g.vh;
    const _Float16* __restrict__ const vl = g.vl;
    extern __shared__ __align__(16) uint32_t wl[];
    uint32_t* const sl = wl + L::kW;
    _Float16* const al = reinterpret_cast<_Float16*>(wl + L::kW + L::kS);  // [part][member][L::kAStride]
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t wr = wave & 1, wk = wave >> 1;
    const uint32_t n16 = lane & 15, kg = lane >> 4;
    __shared__ uint32_t s_row[kMembers];  // the members' act rows
    __shared__ float s_mul[kMembers];     // and the powers of two of their split vectors
    uint32_t rb, m, c_begin, c_end, first = 0;
    const void *pw[kMats], *ps[kMats];
    const WideSet* S = nullptr;
    if constexpr (MODE == kWGemv) {
        rb = blockIdx.x;
        c_begin = blockIdx.y * g.range;
        c_end = c_begin + g.range < cols ? c_begin + g.range : cols;
        first = blockIdx.z * kMembers;
        m = n_vec - first < kMembers ? n_vec - first : kMembers;
        pw[0] = g.w0;
        ps[0] = g.s0;
    } else {
        const uint32_t b = wg, j = b >> 3;
        rb = j % nrb;
        const uint32_t si = (j / nrb) * 8 + (b & 7);
        S = &sets[si];
        m = S->count;
        c_begin = 0;
        c_end = cols;
        if constexpr (MODE == kWGateUp) {
            pw[0] = S->p.gate;
            ps[0] = S->p.gate_scale;
            pw[kMats - 1] = S->p.up;
            ps[kMats - 1] = S->p.up_scale;
        } else {
            pw[0] = S->p.down;
            ps[0] = S->p.down_scale;
        }
        if (si >= *set_count) return;  // the record (stale then) was requested along with the count
    }
    const uint32_t r0 = rb * kMatRows;
    const uint32_t nmt = (m + 15) / 16;  // vector tiles
    // {act row, row of the split vectors} of member j
    auto member = [&](uint32_t j) -> uint2 {
        if constexpr (MODE == kWGemv) {
            const uint32_t i = first + (j < m ? j : m - 1);
            return make_uint2(i, i);
        } else {
            const uint32_t a = S->row[j];
            if constexpr (MODE == kWDown) return make_uint2(a, a);
            // the token of an act row: a / k by the reciprocal (a < 4096, k <= 32), or the
            // shared expert's
            return make_uint2(a, a < n_assign ? (a * g.k_inv) >> 20 : a - n_assign);
        }
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
    // of kNA members)
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
    const uint32_t ac = threadIdx.x % kAUpr, am = threadIdx.x / kAUpr;
    uint32_t aoff[kNA];
#pragma unroll
    for (uint32_t i = 0; i < kNA; ++i) aoff[i] = (member(am + kAStep * i).y * cols + 8 * ac) * 2;
    u32x4 sw[kMats][kNU], sa[kParts][kNA];
    uint32_t ssc[kMats] = {}, sts[kMats] = {};
    // FP4 scales: dword c of row threadIdx.x / kSdw
    constexpr uint32_t kSd = L::kSdw ? L::kSdw : 1;
    const uint32_t s_row_l = threadIdx.x / kSd, s_c = threadIdx.x % kSd;
    auto stage = [&](uint32_t c0) {
        const uint32_t kc = FULL || c_end - c0 >= kChunk ? kChunk : c_end - c0;
        if (FULL || kc == kChunk) {
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
            for (uint32_t i = 0; i < kNA; ++i)
                if (kAStep * i / 16 < nmt) {
                    const auto q = __builtin_amdgcn_raw_buffer_load_b128(rh, static_cast<int>(aoff[i]), static_cast<int>(2 * c0), 0);
                    sa[0][i] = u32x4{q[0], q[1], q[2], q[3]};
                    if constexpr (kParts == 2) {
                        const auto p = __builtin_amdgcn_raw_buffer_load_b128(rl, static_cast<int>(aoff[i]), static_cast<int>(2 * c0), 0);
                        sa[1][i] = u32x4{p[0], p[1], p[2], p[3]};
                    }
                }
        } else {  // a short last chunk: the row's last unit shifted to end with it
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
            for (uint32_t i = 0; i < kNA; ++i)
                if (kAStep * i / 16 < nmt && 8 * ac < kc) {
                    const auto q = __builtin_amdgcn_raw_buffer_load_b128(rh, static_cast<int>(aoff[i]), static_cast<int>(2 * c0), 0);
                    sa[0][i] = u32x4{q[0], q[1], q[2], q[3]};
                    if constexpr (kParts == 2) {
                        const auto p = __builtin_amdgcn_raw_buffer_load_b128(rl, static_cast<int>(aoff[i]), static_cast<int>(2 * c0), 0);
                        sa[1][i] = u32x4{p[0], p[1], p[2], p[3]};
                    }
                }
        }
        if constexpr (TR::kScales) {
#pragma unroll
            for (int t = 0; t < kMats; ++t)
                if (s_row_l < kMatRows && (FULL || s_c < TR::sdw(kc))) {
                    const uint32_t r = r0 + s_row_l < rows ? r0 + s_row_l : rows - 1;
                    ssc[t] = as_global(reinterpret_cast<const uint32_t*>(TR::srow(mt[t], c0) +
                                                                         static_cast<size_t>(r) * TR::spitch(mt[t])))[s_c];
                }
        }
        if constexpr (TR::kTileScale)
#pragma unroll
            for (int t = 0; t < kMats; ++t) sts[t] = TR::tile_scales(mt[t], r0, c0, kc);
    };
    uint32_t ts_cur[kMats] = {};
    auto commit = [&](uint32_t c0) {
        const uint32_t kc = FULL || c_end - c0 >= kChunk ? kChunk : c_end - c0;
        typedef uint32_t u32x2s __attribute__((ext_vector_type(2), aligned(8)));
        typedef uint32_t u32x4s __attribute__((ext_vector_type(4), aligned(16)));
#pragma unroll
        for (int t = 0; t < kMats; ++t) {
            uint32_t* base = wl + t * kMatRows * L::kStride;
            if (FULL || kc == kChunk) {
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
                if (s_row_l < kMatRows) sl[t * kMatRows * kSd + threadIdx.x] = ssc[t];
            ts_cur[t] = sts[t];
        }
#pragma unroll
        for (uint32_t i = 0; i < kNA; ++i)
            if (kAStep * i / 16 < nmt && (FULL || 8 * ac < kc)) {
                _Float16* dst = al + (am + kAStep * i) * L::kAStride + 8 * ac;
                *reinterpret_cast<u32x4s*>(dst) = u32x4s{sa[0][i].x, sa[0][i].y, sa[0][i].z, sa[0][i].w};
                if constexpr (kParts == 2)
                    *reinterpret_cast<u32x4s*>(dst + kMembers * L::kAStride) =
                        u32x4s{sa[1][i].x, sa[1][i].y, sa[1][i].z, sa[1][i].w};
            }
    };
    // [row tile][vector tile]: the running sums of up to kFlush chunks, and of those
    f32x4 acc[kRT][kMT], accl[kRT][kMT], total[kRT][kMT];
#pragma unroll
    for (int a = 0; a < kRT; ++a)
#pragma unroll
        for (int b = 0; b < kMT; ++b) acc[a][b] = accl[a][b] = total[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    // LDS row of this lane in row tile rt, and that tile's matrix
    auto tile_mat = [&](int rt) { return MODE == kWGateUp ? rt / (kRT / 2) : 0; };
    auto tile_row = [&](int rt) {
        return MODE == kWGateUp ? wr * (8u * kRT) + static_cast<uint32_t>(rt % (kRT / 2)) * 16u + n16
                                : wr * (16u * kRT) + static_cast<uint32_t>(rt) * 16u + n16;
    };
    // the products of block b of the chunk with vector tiles 0 .. MT - 1
    auto block = [&](uint32_t b, auto mtc) {
        constexpr int MT = decltype(mtc)::value;
        half8 xh[MT], xl[MT];
#pragma unroll
        for (int v = 0; v < MT; ++v) {
            const _Float16* src = al + (16u * v + n16) * L::kAStride + 32u * b + 8u * kg;
            xh[v] = *reinterpret_cast<const half8*>(src);
            if constexpr (kParts == 2) xl[v] = *reinterpret_cast<const half8*>(src + kMembers * L::kAStride);
        }
#pragma unroll
        for (int rt = 0; rt < kRT; ++rt) {
            const uint32_t lr = tile_mat(rt) * kMatRows + tile_row(rt);
            float sc;
            const half8 bw = TR::get(reinterpret_cast<const uint8_t*>(wl + lr * L::kStride),
                                     reinterpret_cast<const uint8_t*>(sl + lr * kSd), ts_cur[tile_mat(rt)], b, kg, sc);
            f32x4 zh[MT], zl[MT];
            const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int v = 0; v < MT; ++v) zh[v] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh[v], bw, zero, 0, 0, 0);
            if constexpr (kParts == 2)
#pragma unroll
                for (int v = 0; v < MT; ++v) zl[v] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xl[v], bw, zero, 0, 0, 0);
#pragma unroll
            for (int v = 0; v < MT; ++v)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    if constexpr (kParts == 1) {
                        acc[rt][v][q] = __builtin_fmaf(sc, zh[v][q], acc[rt][v][q]);
                    } else if constexpr (kApart) {
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
    for (uint32_t c0 = c_begin; c0 < c_end; c0 += kChunk) {
        const uint32_t kc = FULL || c_end - c0 >= kChunk ? kChunk : c_end - c0;
        __syncthreads();  // the previous chunk's (or set's) LDS reads are done
        commit(c0);
        __syncthreads();
        if (c0 + kChunk < c_end) stage(c0 + kChunk);  // in flight during the products
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        const uint32_t per = FULL ? kChunk / 64 : kc / 64;  // blocks of this wave's half
#pragma unroll 1
        for (uint32_t i = 0; i < per; ++i) {
            const uint32_t b = wk * per + i;
            if (kMT == 1 || nmt > 1) block(b, std::integral_constant<int, kMT>{});
            else block(b, std::integral_constant<int, 1>{});
        }
        if (++pending == kFlush) {
            pending = 0;
#pragma unroll
            for (int a = 0; a < kRT; ++a)
#pragma unroll
                for (int v = 0; v < kMT; ++v) {
                    if constexpr (kApart) acc[a][v] += accl[a][v];
                    total[a][v] += acc[a][v];
                    acc[a][v] = accl[a][v] = f32x4{0.f, 0.f, 0.f, 0.f};
                }
        }
    }
    if (threadIdx.x < kMembers) {
        const uint2 o = member(threadIdx.x);
        s_row[threadIdx.x] = o.x;
        s_mul[threadIdx.x] = g.vmult[o.y];
    }
#pragma unroll
    for (int a = 0; a < kRT; ++a)
#pragma unroll
        for (int v = 0; v < kMT; ++v) {
            if constexpr (kApart) acc[a][v] += accl[a][v];
            total[a][v] += acc[a][v];
        }
    // the two column halves meet in LDS: wave (wr, wk) finishes vector tiles v with
    // v % 2 == wk and hands the others over
    f32x4* const red = reinterpret_cast<f32x4*>(wl) + wr * kRT * kMT * 64;
    __syncthreads();
#pragma unroll
    for (int v = 0; v < kMT; ++v)
        if ((v & 1) != static_cast<int>(wk) && static_cast<uint32_t>(v) < nmt) {
#pragma unroll
            for (int rt = 0; rt < kRT; ++rt) red[(v * kRT + rt) * 64 + lane] = total[rt][v];
        }
    __syncthreads();
    // lane: weight row n16 of the tile, members 16 v + 4 kg + q
#pragma unroll
    for (int v = 0; v < kMT; ++v) {
        if ((v & 1) != static_cast<int>(wk) || static_cast<uint32_t>(v) >= nmt) continue;
#pragma unroll
        for (int rt = 0; rt < kRT; ++rt) total[rt][v] += red[(v * kRT + rt) * 64 + lane];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint32_t j = 16u * v + 4u * kg + static_cast<uint32_t>(q);
            const float mul = s_mul[j];
            const size_t at = MODE == kWGemv ? (static_cast<size_t>(blockIdx.y) * n_vec + s_row[j]) * rows
                                             : static_cast<size_t>(s_row[j]) * rows;
            if constexpr (MODE == kWGateUp) {
#pragma unroll
                for (int h = 0; h < kRT / 2; ++h) {
                    const uint32_t r = r0 + tile_row(h);
                    if (j < m && r < rows)
                        g.out[at + r] = swiglu(total[h][v][q] * mul, total[h + kRT / 2][v][q] * mul, g.limit, g.official);
                }
            } else {
#pragma unroll
                for (int rt = 0; rt < kRT; ++rt) {
                    const uint32_t r = r0 + tile_row(rt);
                    if (j < m && r < rows) g.out[at + r] = total[rt][v][q] * mul;
                }
            }
        }
    }
}

template <class R, class K, int MODE, bool FULL>
__global__ __launch_bounds__(256, K::kWaves) void wide_products_kernel(WideArgs g) {
    wide_body<R, K, MODE, FULL>(g, g.n, g.sets, blockIdx.x);
}

// The official layer's products of a phase: the first n_sh workgroups take the FP8 shared
// expert's sets (few, and the longest rows), the others the routed FP4 experts'. Apart
// they took 37 + 254 us (gate/up) and 20 + 219 us (down) at 32 tokens of hidden 7168.
template <class K, class KS, int MODE, bool FULL>
__global__ __launch_bounds__(256, K::kWaves) void wide_pair_kernel(WideArgs g, const uint32_t* __restrict__ shared_n,
                                                                   const WideSet* __restrict__ shared_sets,
                                                                   uint32_t n_sh, uint32_t shared_nrb) {
    if (blockIdx.x < n_sh) {
        WideArgs h = g;
        h.nrb = shared_nrb;
        wide_body<Fp8Rows, KS, MODE, FULL>(h, shared_n, shared_sets, blockIdx.x);
    } else {
        wide_body<Fp4Rows, K, MODE, FULL>(g, g.n, g.sets, blockIdx.x - n_sh);
    }
}

size_t al256(size_t v) { return (v + 255) & ~size_t(255); }

template <class K, int MODE>
uint32_t row_blocks(uint32_t rows) {
    const uint32_t mr = MODE == kWGateUp ? K::kRows / 2 : K::kRows;
    return (rows + mr - 1) / mr;
}

// Workgroups of a MoE phase: every (row block, set) pair there can be, in whole rounds of
// the eight XCDs; a set's number is below max_sets, the real count is known on the device.
uint32_t phase_blocks(uint32_t nrb, uint32_t max_sets) { return 8 * nrb * ((max_sets + 7) / 8); }

template <class R, class K, int MODE>
void launch_wide_products(hipStream_t s, dim3 grid, const WideArgs& g) {
    const size_t lds = 4 * static_cast<size_t>(WideLds<R, K>::kDwords);
    if (g.cols % K::kChunk == 0)
        hipLaunchKernelGGL((wide_products_kernel<R, K, MODE, true>), grid, dim3(256), lds, s, g);
    else
        hipLaunchKernelGGL((wide_products_kernel<R, K, MODE, false>), grid, dim3(256), lds, s, g);
}

template <class R, class K, int MODE>
void launch_wide_phase(hipStream_t s, WideArgs g, uint32_t max_sets) {
    g.nrb = row_blocks<K, MODE>(g.rows);
    launch_wide_products<R, K, MODE>(s, dim3(phase_blocks(g.nrb, max_sets)), g);
}

template <class K, class KS, int MODE>
void launch_wide_pair(hipStream_t s, WideArgs g, uint32_t max_sets, const uint32_t* shared_n,
                      const WideSet* shared_sets, uint32_t max_shared) {
    g.nrb = row_blocks<K, MODE>(g.rows);
    const uint32_t nrb_s = row_blocks<KS, MODE>(g.rows), n_sh = phase_blocks(nrb_s, max_shared);
    const uint32_t dw = WideLds<Fp4Rows, K>::kDwords > WideLds<Fp8Rows, KS>::kDwords ? WideLds<Fp4Rows, K>::kDwords
                                                                                      : WideLds<Fp8Rows, KS>::kDwords;
    const dim3 grid(n_sh + phase_blocks(g.nrb, max_sets));
    static_assert(K::kChunk == KS::kChunk, "one FULL for both");
    if (g.cols % K::kChunk == 0)
        hipLaunchKernelGGL((wide_pair_kernel<K, KS, MODE, true>), grid, dim3(256), 4 * static_cast<size_t>(dw), s, g,
                           shared_n, shared_sets, n_sh, nrb_s);
    else
        hipLaunchKernelGGL((wide_pair_kernel<K, KS, MODE, false>), grid, dim3(256), 4 * static_cast<size_t>(dw), s, g,
                           shared_n, shared_sets, n_sh, nrb_s);
}

// Offsets in the kernels are 32-bit: matrices and split vectors below 2^31 bytes.
bool below_2g(uint64_t rows, uint64_t bytes_per_row) { return rows * bytes_per_row < (uint64_t(1) << 31); }

// Large work (128 weight rows per workgroup) where the matrices are large and an expert
// has many vectors; 64 rows otherwise (more workgroups, a shorter chain of chunks each).
// us per layer, large / small, each pair on one input: Q4_0 2048 x 768, 128 experts, top-8 at
// 512 tokens 366 / 376, at 200 181 / 178; Q4_0 4096 x 1536, 64 experts at 256 tokens 505 /
// 543, at 40 280 / 233; IQ3_0 2048 x 2048 at 300 tokens 443 / 520; Q4_0 1024 x 512, 16
// experts at 250 tokens 63 / 59. The assignments are the whole call's, not one launch's
// slice of them: 384 experts at 1000 tokens of Q5_0 2048 x 768, top-8, in two launches 904 /
// 932. Split FP4 work items hold 16 vectors in both: from about one vector per expert of
// very large matrices (7168 x 2048, 64 experts, 32 tokens 411 / 435; official, 256 experts,
// 6 tokens 195 / 187).
bool large_work(bool fp4, uint64_t rows, uint64_t cols, uint64_t n_assign, uint64_t n_table) {
    return (n_assign >= 16 * n_table && rows * cols >= (uint64_t(1) << 20)) ||
           (fp4 && n_assign >= n_table && rows * cols >= (uint64_t(8) << 20));
}

uint32_t most_sets(uint32_t a, uint32_t n_table, uint32_t members) { return (a < n_table ? a : n_table) + a / members; }

uint32_t reciprocal(uint64_t k) { return static_cast<uint32_t>(((uint64_t(1) << 20) + k - 1) / k); }

WideArgs gate_up_args(const GroupedWs& w, uint32_t hidden, uint32_t inter, uint64_t k, uint32_t a, float limit, bool official) {
    WideArgs g{};
    g.n = w.hdr;
    g.sets = static_cast<WideSet*>(w.sets);
    g.vh = w.xh;
    g.vl = w.xl;
    g.vmult = w.xmult;
    g.out = w.act;
    g.cols = hidden;
    g.rows = inter;
    g.k_inv = reciprocal(k);
    g.n_assign = a;
    g.limit = limit;
    g.official = official ? 1u : 0u;
    return g;
}

WideArgs down_args(const GroupedWs& w, uint32_t inter, uint32_t out_dim, uint32_t a) {
    WideArgs g{};
    g.n = w.hdr;
    g.sets = static_cast<WideSet*>(w.sets);
    g.vh = w.ah;
    g.vl = w.al;
    g.vmult = w.amult;
    g.out = w.part;
    g.cols = inter;
    g.rows = out_dim;
    g.n_assign = a;
    return g;
}

bool wide_shape(int32_t format, uint64_t n_table, uint64_t k, uint64_t hidden, uint64_t inter, uint64_t out_dim) {
    if (format < OBJETA_HIP_Q4_0 || format > OBJETA_HIP_FP4_E2M1) return false;
    if (k == 0 || k > 32 || n_table == 0 || n_table > kWMaxTable || out_dim == 0) return false;
    if (hidden == 0 || inter == 0 || hidden % 64 || inter % 64 || hidden > (1u << 20) || inter > (1u << 20) ||
        out_dim > (1u << 20))
        return false;
    return format != OBJETA_HIP_FP4_E2M1 || (hidden % 128 == 0 && inter % 128 == 0);
}

}  // namespace

// FP8 is the widest of the formats.
bool matrices_fit(int32_t format, bool official, uint64_t hidden, uint64_t inter, uint64_t out_dim) {
    const uint64_t per32 = official ? 32 : format == OBJETA_HIP_Q4_0 ? 18 : format == OBJETA_HIP_Q5_0 ? 22
                         : format == OBJETA_HIP_IQ3_0 ? 14 : 16;
    return below_2g(inter, hidden / 32 * per32) && below_2g(out_dim, inter / 32 * per32);
}

// Tokens of one launch: at most kWMaxAssign assignments, split vectors below 2^31 bytes.
uint64_t wide_tokens(uint64_t k, uint64_t hidden, uint64_t inter) {
    const uint64_t lim = (uint64_t(1) << 31) - 1;
    uint64_t t = kWMaxAssign / k;
    if (t > lim / (2 * hidden)) t = lim / (2 * hidden);
    if (t > lim / (2 * inter * (k + 1))) t = lim / (2 * inter * (k + 1));
    return t;
}

bool wide_overwrites_x(const float* x, const float* out, uint64_t n_tokens, uint64_t k, uint64_t hidden, uint64_t inter,
                       uint64_t out_dim) {
    if (n_tokens <= wide_tokens(k, hidden, inter)) return false;
    const uintptr_t x0 = reinterpret_cast<uintptr_t>(x), o0 = reinterpret_cast<uintptr_t>(out);
    const bool apart = o0 + 4 * n_tokens * out_dim <= x0 || x0 + 4 * n_tokens * hidden <= o0;
    return !apart && !(o0 <= x0 && out_dim <= hidden);
}

bool wide_supported(int32_t format, uint64_t n_table, uint64_t n_tokens, uint64_t k, uint64_t hidden, uint64_t inter,
                    uint64_t out_dim) {
    if (n_tokens < (format == OBJETA_HIP_FP4_E2M1 ? 1 : kWideMinTokens)) return false;
    // refused by every form, as by the per-assignment kernels
    if (n_tokens > 0x7FFFFFFFull || n_tokens * k * inter > 0x7FFFFFFFull || n_tokens * out_dim > 0x7FFFFFFFull) return false;
    return wide_shape(format, n_table, k, hidden, inter, out_dim) && matrices_fit(format, false, hidden, inter, out_dim) &&
           wide_tokens(k, hidden, inter) > 0;
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
    const uint32_t kk = static_cast<uint32_t>(k), E = static_cast<uint32_t>(n_table);
    const bool fp4 = format == OBJETA_HIP_FP4_E2M1, large = large_work(fp4, inter, hidden, n_tokens * k, n_table);
    const uint32_t M = large && !fp4 ? WorkLarge::kMembers : WorkSmall::kMembers;
    // tokens in equal slices (the workspace of a slice is reused by the next)
    const uint64_t per = wide_tokens(k, hidden, inter), slices = (n_tokens + per - 1) / per;
    const uint64_t slice = (n_tokens + slices - 1) / slices;
    auto sets_of = [&](uint64_t t) {
        return most_sets(static_cast<uint32_t>(t) * kk, E, M) + (shared ? static_cast<uint32_t>((t + M - 1) / M) : 0u);
    };
    // the workspace of the longest slice that a smaller batch can have
    GroupedWs w;
    OBJ_TRY(grouped_workspace(ctx, s, n_tokens < per ? n_tokens : per, k, n_table, shared != nullptr, hidden, inter, out_dim,
                              false, w));
    const bool perm = fp4 ? Tile<Fp4Rows>::kPermuted : Tile<QRows<kQ4>>::kPermuted;
    for (uint64_t t0 = 0; t0 < n_tokens; t0 += slice) {
        const uint32_t t = static_cast<uint32_t>(n_tokens - t0 < slice ? n_tokens - t0 : slice), a = t * kk;
        const uint32_t ns = sets_of(t);
        const uint32_t* idt = ids + t0 * k;
        hipLaunchKernelGGL(wide_prepare_kernel, dim3(1 + t), dim3(256), 0, s, idt, a, E, table, shared, t, M, w.hdr,
                           static_cast<WideSet*>(w.sets), static_cast<WideSet*>(nullptr), ctx->err_word, x + t0 * hidden, H,
                           w.xh, w.xl, w.xmult, perm ? 1u : 0u);
        const WideArgs gu = gate_up_args(w, H, I, k, a, limit, false), dn = down_args(w, I, O, a);
        const uint32_t nr = a + (shared ? t : 0);
#define OBJ_WIDE_LAYER(R, K)                                                                                       \
    {                                                                                                              \
        launch_wide_phase<R, K, kWGateUp>(s, gu, ns);                                                              \
        hipLaunchKernelGGL(wide_split_kernel, dim3(nr), dim3(256), 0, s, w.act, I, w.ah, w.al, w.amult, perm ? 1u : 0u); \
        launch_wide_phase<R, K, kWDown>(s, dn, ns);                                                                \
    }
        switch (format) {
            case OBJETA_HIP_Q4_0:
                if (large) OBJ_WIDE_LAYER(QRows<kQ4>, WorkLarge) else OBJ_WIDE_LAYER(QRows<kQ4>, WorkSmall)
                break;
            case OBJETA_HIP_Q5_0:
                if (large) OBJ_WIDE_LAYER(QRows<kQ5>, WorkLarge) else OBJ_WIDE_LAYER(QRows<kQ5>, WorkSmall)
                break;
            case OBJETA_HIP_IQ3_0:
                if (large) OBJ_WIDE_LAYER(QRows<kIQ3>, WorkLarge) else OBJ_WIDE_LAYER(QRows<kIQ3>, WorkSmall)
                break;
            default:
                if (large) OBJ_WIDE_LAYER(Fp4Rows, WorkLarge4) else OBJ_WIDE_LAYER(Fp4Rows, WorkSmall)
                break;
        }
#undef OBJ_WIDE_LAYER
        launch_moe_combine(s, idt, wts + t0 * k, w.part, shared ? w.part + static_cast<size_t>(a) * O : nullptr,
                           resid ? resid + t0 * out_dim : nullptr, out + t0 * out_dim, t, kk, O, E);
        OBJ_HIP(hipGetLastError(), action);
    }
    return 0;
}

bool official_grouped_supported(uint64_t n_table, uint64_t n_tokens, uint64_t k, uint64_t hidden, uint64_t inter,
                                uint64_t out_dim) {
    if (n_tokens < 2 || !wide_shape(OBJETA_HIP_FP4_E2M1, n_table, k, hidden, inter, out_dim)) return false;
    const uint64_t matrices = 2 * inter * hidden + out_dim * inter;  // an expert's weights
    if (n_tokens < kOfficialGroupedMinTokens &&
        n_tokens * (k * (matrices / 32 * 17) + matrices) <
            (n_tokens == 2 ? kOfficialGroupedReadBytes2 : kOfficialGroupedReadBytes))
        return false;
    return matrices_fit(OBJETA_HIP_FP4_E2M1, true, hidden, inter, out_dim) && n_tokens <= wide_tokens(k, hidden, inter);
}

// The official layer of launch_moe_official_fp4 on the grouped products: x is quantized
// and dequantized as there (its values, a 4-bit significand times a power of two, are
// their own fp16 high part: what lies below 2^-38 of the row's largest value, past the
// fp16 subnormals, is dropped, far below the last bit of the fp32 sums), the routed FP4
// experts and the FP8 shared expert read each matrix once per member set, in one launch
// per phase, the intermediates are quantized in place, and the combine adds w * down in slot order from zero, then the shared
// expert's down.
int32_t launch_moe_official_grouped(objeta_hip_context* ctx, hipStream_t s, const objeta_hip_expert_ptrs* table,
                                    uint64_t n_table, const objeta_hip_expert_ptrs* shared, const uint32_t* ids,
                                    const float* wts, uint64_t n_tokens, uint64_t k, const float* x, float* out,
                                    uint64_t hidden, uint64_t inter, uint64_t out_dim, float limit,
                                    uint8_t* inter_values, uint8_t* inter_scales) {
    const char* action = "launch official FP4 MoE (grouped)";
    // the routed FP4 and the shared FP8 sets multiply the same split activations
    static_assert(Tile<Fp4Rows>::kPermuted == Tile<Fp8Rows>::kPermuted, "one activation order for both tiles");
    if (!official_grouped_supported(n_table, n_tokens, k, hidden, inter, out_dim))
        OBJ_FAIL(kUnsupported, action, "shape outside the grouped official path");
    if (official_few(n_table, n_tokens, k, hidden, inter, out_dim))
        return launch_moe_official_sets(ctx, s, table, n_table, shared, ids, wts, n_tokens, k, x, out, hidden, inter,
                                        out_dim, limit, inter_values, inter_scales);
    const uint32_t T = static_cast<uint32_t>(n_tokens), A = static_cast<uint32_t>(n_tokens * k);
    const uint32_t NR = A + (shared ? T : 0);  // act rows: routed, then shared
    const uint32_t M = WorkOfficial::kMembers;
    const uint32_t NS = most_sets(A, static_cast<uint32_t>(n_table), M), NSS = shared ? (T + M - 1) / M : 0;
    const uint32_t H = static_cast<uint32_t>(hidden), I = static_cast<uint32_t>(inter), O = static_cast<uint32_t>(out_dim);
    GroupedWs w;
    OBJ_TRY(grouped_workspace(ctx, s, T, k, n_table, shared != nullptr, hidden, inter, out_dim, true, w));
    WideSet* const shared_sets = static_cast<WideSet*>(w.shared_sets);
    const bool large = large_work(true, inter, hidden, A, n_table);
    const uint32_t perm = Tile<Fp4Rows>::kPermuted ? 1u : 0u;
    OBJ_TRY(launch_act_quant(s, x, T, H, nullptr, nullptr, w.xd));
    hipLaunchKernelGGL(wide_prepare_kernel, dim3(1 + T), dim3(256), 0, s, ids, A, static_cast<uint32_t>(n_table), table,
                       shared, T, M, w.hdr, static_cast<WideSet*>(w.sets), shared_sets, ctx->err_word, w.xd, H, w.xh,
                       static_cast<_Float16*>(nullptr), w.xmult, perm);
    const WideArgs gu = gate_up_args(w, H, I, k, A, limit, true), dn = down_args(w, I, O, A);
    if (shared) {
        if (large) launch_wide_pair<WorkOfficial, WorkOfficialSmall, kWGateUp>(s, gu, NS, w.hdr + 1, shared_sets, NSS);
        else launch_wide_pair<WorkOfficialSmall, WorkOfficialSmall, kWGateUp>(s, gu, NS, w.hdr + 1, shared_sets, NSS);
    } else {
        if (large) launch_wide_phase<Fp4Rows, WorkOfficial, kWGateUp>(s, gu, NS);
        else launch_wide_phase<Fp4Rows, WorkOfficialSmall, kWGateUp>(s, gu, NS);
    }
    OBJ_HIP(hipGetLastError(), action);
    OBJ_TRY(launch_act_quant(s, w.act, NR, I, inter_values, inter_scales, w.act));
    hipLaunchKernelGGL(wide_split_kernel, dim3(NR), dim3(256), 0, s, w.act, I, w.ah, static_cast<_Float16*>(nullptr),
                       w.amult, perm);
    if (shared) {
        if (large) launch_wide_pair<WorkOfficial, WorkOfficialSmall, kWDown>(s, dn, NS, w.hdr + 1, shared_sets, NSS);
        else launch_wide_pair<WorkOfficialSmall, WorkOfficialSmall, kWDown>(s, dn, NS, w.hdr + 1, shared_sets, NSS);
    } else {
        if (large) launch_wide_phase<Fp4Rows, WorkOfficial, kWDown>(s, dn, NS);
        else launch_wide_phase<Fp4Rows, WorkOfficialSmall, kWDown>(s, dn, NS);
    }
    launch_moe_combine(s, ids, wts, w.part, shared ? w.part + static_cast<size_t>(A) * O : nullptr, nullptr, out, T,
                       static_cast<uint32_t>(k), O, static_cast<uint32_t>(n_table));
    OBJ_HIP(hipGetLastError(), action);
    return 0;
}

bool gemv_wide_supported(int32_t format, uint64_t rows, uint64_t cols, uint64_t batch) {
    return batch >= kGemvWideMinBatch && batch <= 0x7FFFFFFFull && below_2g(rows, cols);
}

namespace {

// Vectors per launch of the batched GEMV: equal multiples of 32 whose two split parts take
// at most 256 MiB (64 vectors at 2^20 columns), so the workspace is bounded however many
// vectors a call brings: 16384 vectors of 4096 columns go in one. (With 64 MiB, 1200 vectors
// of 14336 columns by 4096 rows took 617 us in two launches, 506 in one.)
uint32_t gemv_slice(uint32_t batch, uint32_t cols) {
    const uint32_t most = (64u << 20) / cols / 32 * 32;
    if (batch <= most) return batch;
    const uint32_t n = (batch + most - 1) / most;
    return ((batch + n - 1) / n + 31) / 32 * 32;
}

// The GEMV's workspace: the split vectors of a slice, then partial sums. Several ranges are
// taken only while row blocks x vector groups are below 2 cus, so below 4 cus workgroups in all:
// a bound that does not fall as the batch grows. At least what gemv_mfma_kernel's passes of
// 8 vectors take, which a smaller batch may need under capture.
struct GemvWs {
    size_t xh, xl, part, bytes;
};
template <class K>
GemvWs gemv_layout(uint32_t cus, uint32_t rows, uint32_t cols, uint32_t batch) {
    const uint64_t slice = gemv_slice(batch, cols), ks_max = ((cols + 255) / 256 + 1) / 2;
    const uint64_t tiles = 4ull * cus * K::kMembers * K::kRows, all = ks_max * slice * rows;
    GemvWs w;
    w.xh = al256(4 * slice);
    w.xl = w.xh + al256(2 * slice * cols);
    w.part = w.xl + al256(2 * slice * cols);
    w.bytes = w.part + (ks_max > 1 ? al256(4 * (tiles < all ? tiles : all)) : 0);
    const size_t passes = gemv_passes_bytes(rows, cols, batch);
    if (w.bytes < passes) w.bytes = passes;
    return w;
}

uint32_t cu_count(const objeta_hip_context* ctx) {
    return ctx->info.compute_units > 0 ? static_cast<uint32_t>(ctx->info.compute_units) : 256u;
}

// us, large / small work: Q5_0 14336 x 4096 by 32 vectors 37.5 / 41.8, Q4_0 4096 x 4096
// by 64 25.5 / 24.5, split FP4 5000 x 3584 by 100 36.3 / 34.4
bool gemv_large(uint64_t rows, uint64_t cols, uint64_t batch) {
    return batch > WorkSmall::kMembers && rows * cols >= (uint64_t(1) << 25);
}

template <class R, class K>
int32_t launch_gemv_wide_t(objeta_hip_context* ctx, hipStream_t s, const void* w, const void* ws, const float* x, float* y,
                           uint32_t rows, uint32_t cols, uint32_t batch) {
    const uint32_t cus = cu_count(ctx), nrb = row_blocks<K, kWGemv>(rows), slice = gemv_slice(batch, cols);
    // at most half as many column ranges as the columns have units of 256
    const uint32_t units = (cols + 255) / 256, ks_max = (units + 1) / 2;
    const GemvWs lay = gemv_layout<K>(cus, rows, cols, batch);
    void* wsp = nullptr;
    OBJ_TRY(ensure_workspace(ctx, s, kWsGemv, lay.bytes, &wsp));
    char* b = static_cast<char*>(wsp);
    float* xmult = reinterpret_cast<float*>(b);
    auto* xh = reinterpret_cast<_Float16*>(b + lay.xh);
    auto* xl = reinterpret_cast<_Float16*>(b + lay.xl);
    WideArgs g{};
    g.w0 = w;
    g.s0 = ws;
    g.vh = xh;
    g.vl = xl;
    g.vmult = xmult;
    g.cols = cols;
    g.rows = rows;
    g.nrb = nrb;
    for (uint32_t v0 = 0; v0 < batch; v0 += slice) {
        const uint32_t n = batch - v0 < slice ? batch - v0 : slice, ng = (n + K::kMembers - 1) / K::kMembers;
        // column ranges for about two workgroups per CU, of at least 512 columns
        uint32_t ks = (2 * cus + nrb * ng - 1) / (nrb * ng);
        if (ks > ks_max) ks = ks_max;
        g.range = 256 * ((units + ks - 1) / ks);
        ks = (cols + g.range - 1) / g.range;
        float* const ys = y + static_cast<size_t>(v0) * rows;
        g.out = ks > 1 ? reinterpret_cast<float*>(b + lay.part) : ys;
        g.n_vec = n;
        hipLaunchKernelGGL(wide_split_kernel, dim3(n), dim3(256), 0, s, x + static_cast<size_t>(v0) * cols, cols, xh, xl,
                           xmult, Tile<R>::kPermuted ? 1u : 0u);
        launch_wide_products<R, K, kWGemv>(s, dim3(nrb, ks, ng), g);
        if (ks > 1) launch_gemv_reduce(s, g.out, ys, rows, n, ks);
        OBJ_HIP(hipGetLastError(), "launch batched GEMV (wide)");
    }
    return 0;
}

}  // namespace

size_t gemv_wide_bytes(objeta_hip_context* ctx, int32_t format, uint64_t rows, uint64_t cols, uint64_t batch) {
    const uint32_t R = static_cast<uint32_t>(rows), C = static_cast<uint32_t>(cols), B = static_cast<uint32_t>(batch);
    const uint32_t cus = cu_count(ctx);
    if (!gemv_large(rows, cols, batch)) return gemv_layout<WorkSmall>(cus, R, C, B).bytes;
    return format == OBJETA_HIP_FP4_E2M1 ? gemv_layout<WorkLarge4>(cus, R, C, B).bytes : gemv_layout<WorkLarge>(cus, R, C, B).bytes;
}

int32_t launch_gemv_wide(objeta_hip_context* ctx, hipStream_t s, int32_t format, const void* w, const void* ws,
                         const float* x, float* y, uint64_t rows, uint64_t cols, uint64_t batch) {
    const uint32_t R = static_cast<uint32_t>(rows), C = static_cast<uint32_t>(cols), B = static_cast<uint32_t>(batch);
    const bool large = gemv_large(rows, cols, batch);
#define OBJ_WIDE(RT, KL)                                                                       \
    (large ? launch_gemv_wide_t<RT, KL>(ctx, s, w, ws, x, y, R, C, B)                          \
           : launch_gemv_wide_t<RT, WorkSmall>(ctx, s, w, ws, x, y, R, C, B))
    switch (format) {
        case OBJETA_HIP_Q4_0: return OBJ_WIDE(QRows<kQ4>, WorkLarge);
        case OBJETA_HIP_Q5_0: return OBJ_WIDE(QRows<kQ5>, WorkLarge);
        case OBJETA_HIP_IQ3_0: return OBJ_WIDE(QRows<kIQ3>, WorkLarge);
        default: return OBJ_WIDE(Fp4Rows, WorkLarge4);
    }
#undef OBJ_WIDE
}

}  // namespace objeta

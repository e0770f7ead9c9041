// grouped.hip — the grouped-token expert product on gfx950 matrix cores.
//
// With a batch of tokens, the per-(token, slot) kernels of moe.hip stream an
// expert's matrices once per assignment that selected it. Here the assignments
// are grouped by expert on the device and each selected expert's gate, up and
// down matrices are read once for all of its tokens, the products running on
// MFMA (v_mfma_f32_16x16x32_f16). Per layer:
//
//   moe_prepare_kernel   assignments (token, slot) sorted by expert, stable, cut
//                        into sets of up to 8 per expert; and each token's
//                        activation row -> two fp16 parts (see below)
//   moe_grouped_kernel   per (set, 16 rows): silu(gate x) * (up x) for the set
//   moe_split_kernel     the activations of every assignment
//   moe_grouped_kernel   per (set, 16 rows): down act for every assignment
//   moe_combine_kernel   out = residual + sum_j w_j down_j in slot order
//
// Exactness. Weights enter the MFMA as fp16 values that are exact for every
// format: q-8 (Q4_0), q-16 (Q5_0), q-4 (IQ3_0), the E2M1 value * 2^-14 (FP4). The
// block scale multiplies the fp32 block sum. An activation row x is scaled by a
// power of two 2^s (|x 2^s| < 2^14, exact) and split x 2^s = hi + lo with hi, lo
// fp16: hi + lo carries 22 significant bits of x, every weight * part product is
// exact in fp32 and the MFMA accumulates in fp32. The result is within the fp32
// tolerance of the reference's sequential sums (not bit-identical: the order of
// the additions differs, as in every parallel kernel here).
//
// Layout trick: within each 8-element k group the weights of the block formats come
// out of the nibble unpacking as (w0,w4),(w1,w5),(w2,w6),(w3,w7); for them the split
// activations are stored in that same order, so no unpacking shuffle is needed (a k
// permutation applied to both operands leaves the products unchanged). FP4 (the
// hardware conversion's pairs) and FP8 weights come in element order, and so do
// their split activations.
//
// The sets of 8 take the block formats up to 8 tokens and any format's batches of few
// assignments (few_assignments); the others run in wide.hip.
//
// MFMA roles (D = A B, 16x16x32): A = activation parts, row m = 2 * token + part
// (8 tokens per instruction); B = weights, column n = output row. Lane l holds
// B[k = 8(l/16) .. +7][n = l%16] and D[m = 4(l/16) + i][n = l%16]: every lane
// owns one output row, so the block scale it applies is its own row's and the hi
// and lo parts of a token land in the same lane (i = 2q, 2q+1).
//
// Reference: execute_selected_moe_cuda (crates/objeta-cuda/src/moe.rs:352-751)
// runs each selected expert per token; its combine adds w * down in selection
// order (moe.rs:1319-1321), which moe_combine_kernel keeps.
#include "mfma_tiles.hpp"

namespace objeta {
namespace {

using namespace dev;

constexpr uint32_t kGMaxTable = 1024;   // experts per table
constexpr uint32_t kGMaxAssign = 1024;  // tokens * k per call

// One work item of the grouped products: up to 8 assignments (token, slot) that
// selected the same expert, with that expert's table entry copied in, so a
// workgroup reaches its weights and activations through one load.
struct SetRec {
    objeta_hip_expert_ptrs p;
    uint16_t mem[8];  // act rows: assignments t*k + j (in order), or n_assign + t for the
                      // shared expert; unused slots repeat the last; mem[0] bits
                      // 12..15 hold the member count - 1
};
static_assert(sizeof(SetRec) == 64, "one 64-byte record per set");

struct GroupWs {
    uint32_t* hdr;  // [0] number of groups, [1] number of member sets
    SetRec* sets;   // [A] (a set holds at least one assignment)
};

// ------------------------------------------------------------------ grouping
// The shared expert (when given) follows as one more group: member t is token t, its act
// row n_assign + t. Its member sets go after the routed ones in w, or, when wsh.hdr is set
// (a shared expert of another format, multiplied by a launch of its own), into wsh.
__device__ void group_assignments(const uint32_t* __restrict__ ids, uint32_t n_assign, uint32_t n_table,
                                  const objeta_hip_expert_ptrs* __restrict__ table,
                                  const objeta_hip_expert_ptrs* __restrict__ shared, uint32_t n_tokens, GroupWs w,
                                  GroupWs wsh, uint32_t* __restrict__ err) {
    __shared__ uint32_t cnt[kGMaxTable];
    __shared__ uint32_t pos[kGMaxTable];
    __shared__ uint32_t sid[kGMaxAssign];
    __shared__ uint32_t sal[kGMaxAssign];   // assignments grouped by expert
    __shared__ uint32_t sinfo[kGMaxAssign];  // set: expert | first member << 11 | (count - 1) << 22
    __shared__ uint32_t wtot[3][4];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (uint32_t e = tid; e < n_table; e += 256) cnt[e] = 0;
    for (uint32_t a = tid; a < n_assign; a += 256) sid[a] = ids[a];
    __syncthreads();
    bool bad = false;
    for (uint32_t a = tid; a < n_assign; a += 256) {
        if (sid[a] < n_table) atomicAdd(&cnt[sid[a]], 1u);
        else bad = true;
    }
    if (bad) atomicOr(err, 1u);
    __syncthreads();
    // exclusive prefix over experts of the counts (positions), of the non-empty
    // flags (group numbers) and of the member sets; thread t owns experts
    // [t*per, (t+1)*per)
    const uint32_t per = (n_table + 255) / 256;
    const uint32_t e0 = tid * per < n_table ? tid * per : n_table;
    const uint32_t e1 = e0 + per < n_table ? e0 + per : n_table;
    uint32_t sc = 0, sg = 0, ss = 0;
    for (uint32_t e = e0; e < e1; ++e) {
        sc += cnt[e];
        sg += cnt[e] ? 1u : 0u;
        ss += (cnt[e] + 7) / 8;
    }
    uint32_t ic = sc, ig = sg, is = ss;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t oc = __shfl_up(ic, off, 64), og = __shfl_up(ig, off, 64), os = __shfl_up(is, off, 64);
        if (static_cast<int>(lane) >= off) {
            ic += oc;
            ig += og;
            is += os;
        }
    }
    if (lane == 63) {
        wtot[0][wave] = ic;
        wtot[1][wave] = ig;
        wtot[2][wave] = is;
    }
    __syncthreads();
    uint32_t bc = 0, bs = 0, tg = 0, ts = 0;
    for (uint32_t v = 0; v < 4; ++v) {
        if (v < wave) {
            bc += wtot[0][v];
            bs += wtot[2][v];
        }
        tg += wtot[1][v];
        ts += wtot[2][v];
    }
    uint32_t pc = bc + ic - sc, ps = bs + is - ss;
    for (uint32_t e = e0; e < e1; ++e) {
        if (cnt[e]) {
            pos[e] = pc;
            for (uint32_t j = 0; j < cnt[e]; j += 8) {
                const uint32_t m = cnt[e] - j < 8 ? cnt[e] - j : 8;
                sinfo[ps++] = e | ((pc + j) << 11) | ((m - 1) << 22);
            }
            pc += cnt[e];
        }
    }
    const uint32_t n_sh = shared ? (n_tokens + 7) / 8 : 0;
    const bool apart = wsh.hdr != nullptr;
    if (tid == 0) {
        w.hdr[0] = tg + (shared && !apart ? 1 : 0);
        w.hdr[1] = ts + (apart ? 0 : n_sh);
        if (apart) {
            wsh.hdr[0] = shared ? 1 : 0;
            wsh.hdr[1] = n_sh;
        }
    }
    __syncthreads();
    // stable order inside a group: rank among the earlier assignments of the expert
    for (uint32_t a = tid; a < n_assign; a += 256) {
        const uint32_t e = sid[a];
        if (e >= n_table) continue;
        uint32_t r = 0;
        for (uint32_t b = 0; b < a; ++b) r += sid[b] == e ? 1u : 0u;
        sal[pos[e] + r] = a;
    }
    __syncthreads();
    for (uint32_t si = tid; si < ts + n_sh; si += 256) {
        // the record: the expert's table entry, then 8 uint16 act rows (4 dwords),
        // written field by field (a record assembled in a local lands in scratch)
        const objeta_hip_expert_ptrs* src;
        uint32_t first, m1;
        if (si < ts) {
            const uint32_t info = sinfo[si];
            src = table + (info & 0x7FFu);
            first = (info >> 11) & 0x7FFu;
            m1 = info >> 22;
        } else {
            const uint32_t t0 = 8 * (si - ts);
            src = shared;
            first = t0;
            m1 = (n_tokens - t0 < 8 ? n_tokens - t0 : 8) - 1;
        }
        auto row = [&](uint32_t j) {
            const uint32_t jj = j < m1 ? j : m1;
            return si < ts ? sal[first + jj] : n_assign + first + jj;
        };
        uint4 mem;
        mem.x = (row(0) | (m1 << 12)) | (row(1) << 16);
        mem.y = row(2) | (row(3) << 16);
        mem.z = row(4) | (row(5) << 16);
        mem.w = row(6) | (row(7) << 16);
        SetRec* dst = si >= ts && apart ? &wsh.sets[si - ts] : &w.sets[si];
        dst->p = *src;
        *reinterpret_cast<uint4*>(dst->mem) = mem;
    }
}

// Block 0 groups the assignments; block 1 + t splits row t of x.
__global__ __launch_bounds__(256) void moe_prepare_kernel(const uint32_t* __restrict__ ids, uint32_t n_assign,
                                                          uint32_t n_table,
                                                          const objeta_hip_expert_ptrs* __restrict__ table,
                                                          const objeta_hip_expert_ptrs* __restrict__ shared,
                                                          uint32_t n_tokens, GroupWs w, GroupWs wsh,
                                                          uint32_t* __restrict__ err, const float* __restrict__ x,
                                                          uint32_t cols, _Float16* __restrict__ xh,
                                                          _Float16* __restrict__ xl, float* __restrict__ xmult,
                                                          uint32_t perm) {
    if (blockIdx.x == 0) group_assignments(ids, n_assign, n_table, table, shared, n_tokens, w, wsh, err);
    else split_row(x, cols, xh, xl, xmult, blockIdx.x - 1, perm);
}

// One workgroup per row.
__global__ __launch_bounds__(256) void moe_split_kernel(const float* __restrict__ src, uint32_t cols,
                                                        _Float16* __restrict__ hi, _Float16* __restrict__ lo,
                                                        float* __restrict__ mult, uint32_t perm) {
    split_row(src, cols, hi, lo, mult, blockIdx.x, perm);
}


// ----------------------------------------------------------- grouped GEMMs
// A workgroup streams a 16-row slab of one group's expert (gate and up together,
// or down) through LDS in chunks of Tile<R>::kChunkGU / kChunkDn columns, double-buffered: while its
// four waves multiply chunk c (wave w: the w-th quarter of the chunk's blocks), the
// loads of chunk c+1 (every thread's share, 64-byte runs within rows) and the next
// activation operands are already in flight. Each lane takes its MFMA operand (8
// weights of one output row) and the block scale from LDS; the four waves' partial
// sums meet in LDS at the end. 8 group members per MFMA column set; the member
// sets of all groups are separate work items (a larger group's sets stream the slab
// in parallel workgroups).

// A slab's row segments of a chunk (seg dwords per row, at most kSeg) move in 16-byte
// units: unit c of a row covers dwords [min(4c, seg - 4), +4) (seg >= 4 for every
// chunk width and format), so a short last chunk reads inside its rows; thread t takes
// units t, t + 256, ... of the 16 rows in row order. Rows past `rows` read the last
// row. In LDS a row takes kSeg + 4 dwords (16-byte rows; a stride of 12 mod 64 dwords
// spreads the 16 rows x 4 k groups of an MFMA operand read over distinct banks).
template <uint32_t kSeg>
struct SlabUnits {
    static constexpr uint32_t kUpr = (kSeg + 3) / 4;                 // units per row of a full chunk
    static constexpr uint32_t kN = (kSlab * kUpr + 255) / 256;        // units per thread
    static constexpr uint32_t kStride = kSeg + 4;                      // LDS dwords per row
};
// This thread's units of a slab: row byte offsets (rows past `rows` read the last row)
// and unit indices, fixed for a member set.
template <uint32_t kSeg>
struct SlabLanes {
    uint32_t off[SlabUnits<kSeg>::kN];  // byte offset of the unit in a full chunk
    uint32_t c[SlabUnits<kSeg>::kN];    // unit index in its row (0xFFFF: none)
    __device__ __forceinline__ void init(uint32_t r0, uint32_t rows, size_t pitch) {
        using SU = SlabUnits<kSeg>;
#pragma unroll
        for (uint32_t i = 0; i < SU::kN; ++i) {
            const uint32_t u = threadIdx.x + 256u * i;
            const uint32_t rr = u / SU::kUpr;
            c[i] = rr < kSlab ? u - rr * SU::kUpr : 0xFFFFu;
            const uint32_t r = r0 + rr < rows ? r0 + rr : rows - 1;
            off[i] = static_cast<uint32_t>(static_cast<size_t>(r) * pitch) + 16u * (c[i] & 0xFFFu);
        }
    }
};
template <uint32_t kSeg, bool FULL>
__device__ __forceinline__ void slab_load4(__amdgpu_buffer_rsrc_t rs, uint32_t chunk_off, const SlabLanes<kSeg>& ln,
                                           uint32_t seg, u32x4 (&v)[SlabUnits<kSeg>::kN]) {
    using SU = SlabUnits<kSeg>;
    if (FULL || seg == kSeg) {  // a full chunk: the precomputed offsets as they are
#pragma unroll
        for (uint32_t i = 0; i < SU::kN; ++i) {
            if (SU::kN * 256u == kSlab * SU::kUpr || ln.c[i] < SU::kUpr) {
                const auto q = __builtin_amdgcn_raw_buffer_load_b128(rs, static_cast<int>(ln.off[i]),
                                                                     static_cast<int>(chunk_off), 0);
                v[i] = u32x4{q[0], q[1], q[2], q[3]};
            }
        }
        return;
    }
    const uint32_t upr = (seg + 3) / 4;
#pragma unroll
    for (uint32_t i = 0; i < SU::kN; ++i) {
        if (ln.c[i] < upr) {
            const uint32_t d = 4 * ln.c[i] < seg - 4 ? 4 * ln.c[i] : seg - 4;
            const auto q = __builtin_amdgcn_raw_buffer_load_b128(rs, static_cast<int>(ln.off[i] - 16u * ln.c[i] + 4u * d),
                                                                 static_cast<int>(chunk_off), 0);
            v[i] = u32x4{q[0], q[1], q[2], q[3]};
        }
    }
}
template <uint32_t kSeg, bool FULL>
__device__ __forceinline__ void slab_store4(uint32_t* lds, uint32_t seg, const u32x4 (&v)[SlabUnits<kSeg>::kN]) {
    using SU = SlabUnits<kSeg>;
    const uint32_t upr = (seg + 3) / 4;
#pragma unroll
    for (uint32_t i = 0; i < SU::kN; ++i) {
        const uint32_t u = threadIdx.x + 256u * i;
        const uint32_t rr = u / SU::kUpr, c = u - rr * SU::kUpr;
        if (rr < kSlab && c < upr) {
            uint32_t* dst = lds + rr * SU::kStride;
            if (FULL || seg == kSeg) {  // a full chunk: aligned 16-byte stores
                typedef uint32_t u32x4s __attribute__((ext_vector_type(4), aligned(16)));
                *reinterpret_cast<u32x4s*>(dst + 4 * c) = u32x4s{v[i].x, v[i].y, v[i].z, v[i].w};
            } else {
                const uint32_t d = 4 * c < seg - 4 ? 4 * c : seg - 4;
                dst[d] = v[i].x; dst[d + 1] = v[i].y; dst[d + 2] = v[i].z; dst[d + 3] = v[i].w;
            }
        }
    }
}
// FP4 scale rows (seg <= 16 dwords): one dword per thread, thread t row t / 16.
__device__ __forceinline__ void scale_load(const uint8_t* base, size_t pitch, uint32_t r0, uint32_t rows, uint32_t seg,
                                           uint32_t& v) {
    const uint32_t rr = threadIdx.x >> 4, c = threadIdx.x & 15;
    const uint32_t r = r0 + rr < rows ? r0 + rr : rows - 1;
    if (c < seg) v = as_global(reinterpret_cast<const uint32_t*>(base + static_cast<size_t>(r) * pitch))[c];
}
__device__ __forceinline__ void scale_store(uint32_t* lds, uint32_t stride, uint32_t seg, uint32_t v) {
    const uint32_t rr = threadIdx.x >> 4, c = threadIdx.x & 15;
    if (c < seg) lds[rr * stride + c] = v;
}

// One chunk's staged bytes of every matrix of the workgroup, in registers.
template <class R, int M, uint32_t CH>
struct Staged {
    static constexpr uint32_t kSeg = Tile<R>::wdw(CH);
    u32x4 w[M][SlabUnits<kSeg>::kN];
    uint32_t s[M];   // FP4 scales: CH / 128 <= 16 dwords per row
    uint32_t ts[M];  // FP8 tile scales of the chunk
};

// grid = (ceil(rows / 16), gy), 256 threads; workgroup (x, y) takes member sets y,
// y + gy, ... (the number of sets is known only on the device). GATEUP: rows = inter
// over the split x rows (cols = hidden), writes act (the official SwiGLU when `official` is
// set); else rows = out_dim over the split act rows (cols = inter), writes part. Dynamic LDS: two chunk buffers of every matrix.
template <class R, bool GATEUP, bool FULL>
__global__ __launch_bounds__(256) void moe_grouped_kernel(GroupWs gw, const _Float16* __restrict__ vh,
                                                          const _Float16* __restrict__ vl,
                                                          const float* __restrict__ vmult, float* __restrict__ out,
                                                          uint32_t cols, uint32_t rows, uint32_t k, uint32_t n_assign,
                                                          float limit, uint32_t official) {
    extern __shared__ uint32_t tl[];
    // the cross-wave partial sums reuse the chunk buffers once a set's products are done
    auto red = reinterpret_cast<f32x4 (*)[3][64]>(tl);
    constexpr int kMats = GATEUP ? 2 : 1;
    constexpr uint32_t kChunk = GATEUP ? Tile<R>::kChunkGU : Tile<R>::kChunkDn;
    constexpr int kB = kChunk / 32 / 4;  // blocks per wave and chunk
    constexpr uint32_t kSeg = Tile<R>::wdw(kChunk);           // weight dwords per row of a full chunk
    constexpr uint32_t kWStride = SlabUnits<kSeg>::kStride;    // LDS dwords per staged weight row
    constexpr uint32_t kSStride = Tile<R>::sdw(kChunk) + 1;    // LDS dwords per staged scale row (FP4)
    static_assert(Tile<R>::lds_dw(kChunk) == kSlab * kWStride + (Tile<R>::kScales ? kSlab * kSStride : 0u),
                  "LDS chunk layout");
    const uint32_t n_sets = gw.hdr[1];
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t r0 = blockIdx.x * kSlab;
    const uint32_t row = r0 + (lane & 15), kg = lane >> 4;
    const uint32_t nchunks = (cols + kChunk - 1) / kChunk;
    const uint32_t buf_dw = kMats * Tile<R>::lds_dw(kChunk);
    for (uint32_t si = blockIdx.y; si < n_sets; si += gridDim.y) {
        const SetRec sr = gw.sets[si];
        const objeta_hip_expert_ptrs& P = sr.p;
        const uint32_t m = (sr.mem[0] >> 12) + 1u;
        auto member = [&](uint32_t j) {  // assignment of member j (< 8)
            uint32_t a = sr.mem[0] & 0xFFFu;
#pragma unroll
            for (uint32_t q = 1; q < 8; ++q) a = j == q ? sr.mem[q] : a;
            return a;
        };
        R mt[kMats];
        mt[0] = GATEUP ? RowsOf<R>::make(P.gate, P.gate_scale, cols) : RowsOf<R>::make(P.down, P.down_scale, cols);
        if constexpr (GATEUP) mt[kMats - 1] = RowsOf<R>::make(P.up, P.up_scale, cols);
        const size_t wpitch = Tile<R>::wpitch(mt[0]), spitch = Tile<R>::spitch(mt[0]);
        SlabLanes<kSeg> lanes;
        lanes.init(r0, rows, wpitch);
        __amdgpu_buffer_rsrc_t rs[kMats];
#pragma unroll
        for (int t = 0; t < kMats; ++t) rs[t] = matrix_rsrc(Tile<R>::wrow(mt[t], 0));
        // A operand rows: member (lane&15)/2 of the set, part (lane&1)
        const uint32_t am = member((lane & 15) >> 1);
        // token row of x (routed or shared act row), or the act row itself
        auto xrow = [&](uint32_t a) { return a < n_assign ? a / k : a - n_assign; };
        const uint32_t vrow = GATEUP ? xrow(am) : am;
        auto stage = [&](uint32_t kc0, Staged<R, kMats, kChunk>& st) {
            const uint32_t kc = FULL ? kChunk : (cols - kc0 < kChunk ? cols - kc0 : kChunk);
#pragma unroll
            for (int t = 0; t < kMats; ++t) {
                slab_load4<kSeg, FULL>(rs[t], static_cast<uint32_t>(Tile<R>::wrow(mt[t], kc0) - Tile<R>::wrow(mt[t], 0)), lanes,
                                 Tile<R>::wdw(kc), st.w[t]);
                if constexpr (Tile<R>::kScales)
                    scale_load(Tile<R>::srow(mt[t], kc0), spitch, r0, rows, Tile<R>::sdw(kc), st.s[t]);
                if constexpr (Tile<R>::kTileScale) st.ts[t] = Tile<R>::tile_scales(mt[t], r0, kc0, kc);
            }
        };
        uint32_t ts_cur[kMats] = {};  // the tile scales of the chunk being multiplied
        auto operands = [&](uint32_t kc0, half8 (&xr)[kB]) {
            const uint32_t kc = FULL ? kChunk : (cols - kc0 < kChunk ? cols - kc0 : kChunk);
            const uint32_t nb = kc / 32, per = (nb + 3) / 4;
            const uint32_t b0 = wave * per < nb ? wave * per : nb, b1 = b0 + per < nb ? b0 + per : nb;
#pragma unroll
            for (int i = 0; i < kB; ++i) {
                const uint32_t b = b0 + static_cast<uint32_t>(i) < b1 ? b0 + static_cast<uint32_t>(i) : (b1 ? b1 - 1 : 0);
                const size_t at = static_cast<size_t>(vrow) * cols + kc0 + 32 * b + 8 * kg;
                xr[i] = *as_global(reinterpret_cast<const half8*>(((lane & 1) ? vl : vh) + at));
            }
        };
        auto commit = [&](uint32_t kc0, uint32_t buf, const Staged<R, kMats, kChunk>& st) {
            const uint32_t kc = FULL ? kChunk : (cols - kc0 < kChunk ? cols - kc0 : kChunk);
#pragma unroll
            for (int t = 0; t < kMats; ++t) {
                uint32_t* base = tl + buf * buf_dw + t * Tile<R>::lds_dw(kChunk);
                slab_store4<kSeg, FULL>(base, Tile<R>::wdw(kc), st.w[t]);
                if constexpr (Tile<R>::kScales)
                    scale_store(base + kSlab * kWStride, kSStride, Tile<R>::sdw(kc), st.s[t]);
                // read only after the products of the previous chunk
                if constexpr (Tile<R>::kTileScale) ts_cur[t] = st.ts[t];
            }
        };
        f32x4 acc[kMats];
#pragma unroll
        for (int t = 0; t < kMats; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
        Staged<R, kMats, kChunk> st;
        half8 xa[kB];
        stage(0, st);
        operands(0, xa);
        commit(0, 0, st);
        __syncthreads();
        for (uint32_t c = 0; c < nchunks; ++c) {
            const uint32_t kc0 = c * kChunk;
            const uint32_t kc = FULL ? kChunk : (cols - kc0 < kChunk ? cols - kc0 : kChunk);
            if (c + 1 < nchunks) stage(kc0 + kChunk, st);  // in flight during the products below
            asm volatile("" ::: "memory");  // the loads stay ahead of the products
            __builtin_amdgcn_sched_barrier(0);
            const uint32_t nb = kc / 32, per = (nb + 3) / 4;
            const uint32_t b0 = wave * per < nb ? wave * per : nb, b1 = b0 + per < nb ? b0 + per : nb;
#pragma unroll
            for (int t = 0; t < kMats; ++t) {
                const uint32_t* base = tl + (c & 1) * buf_dw + t * Tile<R>::lds_dw(kChunk);
                const uint8_t* wl = reinterpret_cast<const uint8_t*>(base + (lane & 15) * kWStride);
                const uint8_t* sl = reinterpret_cast<const uint8_t*>(base + kSlab * kWStride + (lane & 15) * kSStride);
                f32x4 part = {0.f, 0.f, 0.f, 0.f};  // of this chunk: short chains round less
#pragma unroll
                for (int i = 0; i < kB; ++i) {
                    if (b0 + static_cast<uint32_t>(i) >= b1) break;
                    float sc;
                    const half8 bw = Tile<R>::get(wl, sl, ts_cur[t], b0 + static_cast<uint32_t>(i), kg, sc);
                    const f32x4 z = {0.f, 0.f, 0.f, 0.f};
                    const f32x4 r = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[i], bw, z, 0, 0, 0);
#pragma unroll
                    for (int q = 0; q < 4; ++q) part[q] = __builtin_fmaf(sc, r[q], part[q]);
                }
                acc[t] += part;
                // added here and not after both matrices' products, which keeps four registers
                // fewer alive (split FP4 gate/up 126, not 130: four waves per SIMD; hidden 7168,
                // top-2 at 8 tokens 81 against 94 us)
                asm volatile("" : "+v"(acc[t]));
            }
            if (c + 1 < nchunks) {
                // the next activation operands (into the registers just used) travel
                // while the staged weights are stored; buffer (c+1)&1 was last read in
                // iteration c-1, which every wave has finished (the barrier below)
                operands(kc0 + kChunk, xa);
                commit(kc0 + kChunk, (c + 1) & 1, st);
            }
            __syncthreads();
        }
        // the four waves' partial sums (same lane layout) meet in LDS; wave 0 adds
        if (wave > 0) {
#pragma unroll
            for (int t = 0; t < kMats; ++t) red[t][wave - 1][lane] = acc[t];
        }
        __syncthreads();
        if (wave == 0) {
#pragma unroll
            for (int t = 0; t < kMats; ++t) acc[t] = (acc[t] + red[t][0][lane]) + (red[t][1][lane] + red[t][2][lane]);
            // lane: output row `row`, members 2kg + q (q = 0, 1) as (hi, lo) in 2q, 2q+1
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const uint32_t j = 2 * kg + static_cast<uint32_t>(q);  // uniform over 16 lanes
                const bool live = j < m && row < rows;
                const uint32_t a = member(j);  // unused slots repeat the last member
                const float mul = vmult[GATEUP ? xrow(a) : a];
                const float v0 = (acc[0][2 * q] + acc[0][2 * q + 1]) * mul;
                if constexpr (GATEUP) {
                    const float v1 = (acc[kMats - 1][2 * q] + acc[kMats - 1][2 * q + 1]) * mul;
                    if (live) out[static_cast<size_t>(a) * rows + row] = swiglu(v0, v1, limit, official);
                } else {
                    if (live) out[static_cast<size_t>(a) * rows + row] = v0;
                }
            }
        }
        __syncthreads();  // red is reused by the next member set
    }
}

// ------------------------------------------------------ batched GEMV on MFMA
// y[b][r] = sum_c W[r][c] x[b][c] for up to 8 vectors at once: the grouped
// products' down form with the matrix as the one expert and the vectors as the
// members, so every weight is decoded once for all of them. A workgroup covers
// S slabs of 16 rows over the column range [y * kGemvRange, (y + 1) * kGemvRange):
//   1. every thread issues its share of the tile's weight loads (the whole tile is
//      in flight at once: an 8-vector GEMV is a few MB to a few tens of MB, and the
//      loads in flight, not the arithmetic, set its time at these sizes);
//   2. meanwhile it splits that slice of every vector into two fp16 parts in LDS
//      (with the slice's own power of two, which the partial sums take back): the
//      split is shared by the 16 S rows of the workgroup;
//   3. the weights go to LDS, one row per padded LDS row;
//   4. wave w multiplies slabs w, w + 4, ... over every block of the range (no
//      barrier inside the loop, no cross-wave sum) and writes the partial sums of
//      its rows to part[range][b][r]; gemv_reduce_kernel adds the ranges in order.
constexpr uint32_t kGemvRange = 512;               // columns per workgroup
constexpr uint32_t kGemvXStride = kGemvRange + 8;  // halves per staged vector part (padded)

typedef uint32_t u32x4a __attribute__((ext_vector_type(4), aligned(16)));

// LDS layout of a tile: 16 S rows of kWStride dwords (a full range's row segment,
// padded to keep 16-byte rows), then, for the split FP4 layout, 16 S rows of
// kSStride dwords of E8M0 scales.
template <class R, int S>
struct GemvTile {
    static constexpr uint32_t kRows = 16u * S;
    static constexpr uint32_t kWdw = Tile<R>::wdw(kGemvRange);
    static constexpr uint32_t kWStride = kWdw + 4;
    static constexpr uint32_t kSdw = Tile<R>::kScales ? Tile<R>::sdw(kGemvRange) : 0u;
    static constexpr uint32_t kSStride = Tile<R>::kScales ? kSdw + 1 : 0u;
    static constexpr size_t lds_bytes() { return 4ull * kRows * (kWStride + kSStride); }
};

// Weight units of V dwords (V = 4: 16-byte rows and range starts, every range full;
// V = 1: any 4-byte aligned layout, the last range possibly short).
template <int V>
struct WUnit;
template <>
struct WUnit<4> {
    typedef u32x4a T;
    static __device__ __forceinline__ T load(gptr<uint32_t> p) { return *(gptr<u32x4a>)(p); }
};
template <>
struct WUnit<1> {
    typedef uint32_t T;
    static __device__ __forceinline__ T load(gptr<uint32_t> p) { return *p; }
};

template <class R, int S, int V>
__global__ __launch_bounds__(256) void gemv_mfma_kernel(const void* __restrict__ w, const void* __restrict__ ws,
                                                        const float* __restrict__ x, float* __restrict__ part,
                                                        uint32_t rows, uint32_t cols, uint32_t n_vec) {
    using TL = GemvTile<R, S>;
    using U = typename WUnit<V>::T;
    extern __shared__ __align__(16) uint32_t tl[];
    __shared__ __align__(16) _Float16 xs[2][8][kGemvXStride];  // [hi / lo][vector][column of the range]
    __shared__ float xmul[8];
    constexpr uint32_t kUpr = TL::kWdw / V;                  // units per row of a full range
    constexpr uint32_t kNU = (TL::kRows * kUpr + 255) / 256;  // units per thread
    constexpr uint32_t kSUpr = TL::kSdw;                      // scale dwords per row (FP4)
    constexpr uint32_t kNS = (TL::kRows * kSUpr + 255) / 256;
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t r0 = blockIdx.x * TL::kRows;
    const uint32_t k0 = blockIdx.y * kGemvRange, k1 = k0 + kGemvRange < cols ? k0 + kGemvRange : cols;
    const uint32_t kc = k1 - k0;
    const uint32_t wdw = Tile<R>::wdw(kc);  // dwords of this range's row segments
    const R mt = RowsOf<R>::make(w, ws, cols);
    // 1. the vectors' slices (32 threads per vector, 16 consecutive columns each), then
    // the tile's weight (and scale) loads, all in flight together (the split below
    // waits for the slices alone)
    const uint32_t xb = threadIdx.x >> 5, xc = (threadIdx.x & 31) * 16;
    const bool xlive = xb < n_vec && k0 + xc < k1;
    float v[16];
    if (xlive) {
        const gptr<f32x4> src = as_global(reinterpret_cast<const f32x4*>(x + static_cast<size_t>(xb) * cols + k0 + xc));
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const f32x4 f = src[q];
            v[4 * q] = f[0]; v[4 * q + 1] = f[1]; v[4 * q + 2] = f[2]; v[4 * q + 3] = f[3];
        }
    }
    // rows past `rows` read the last row, units past the range's end are not read
    U wv[kNU];
    {
        const uint8_t* wb = Tile<R>::wrow(mt, k0);
        const size_t pitch = Tile<R>::wpitch(mt);
#pragma unroll
        for (uint32_t i = 0; i < kNU; ++i) {
            const uint32_t u = threadIdx.x + 256u * i;
            const uint32_t rr = u / kUpr, c = u - rr * kUpr;
            if (rr < TL::kRows && c * V < wdw) {
                const uint32_t r = r0 + rr < rows ? r0 + rr : rows - 1;
                wv[i] = WUnit<V>::load(as_global(reinterpret_cast<const uint32_t*>(wb + static_cast<size_t>(r) * pitch)) + c * V);
            }
        }
    }
    uint32_t sv[kNS > 0 ? kNS : 1];
    if constexpr (kNS > 0) {
        const uint8_t* sb = Tile<R>::srow(mt, k0);
        const size_t spitch = Tile<R>::spitch(mt);
        const uint32_t sdw = Tile<R>::sdw(kc);
#pragma unroll
        for (uint32_t i = 0; i < kNS; ++i) {
            const uint32_t u = threadIdx.x + 256u * i;
            const uint32_t rr = u / kSUpr, c = u - rr * kSUpr;
            if (rr < TL::kRows && c < sdw) {
                const uint32_t r = r0 + rr < rows ? r0 + rr : rows - 1;
                sv[i] = as_global(reinterpret_cast<const uint32_t*>(sb + static_cast<size_t>(r) * spitch))[c];
            }
        }
    }
    // 2. the slices split into two fp16 parts (the slice's power of two in xmul)
    {
        const uint32_t b = xb, c = xc;
        const bool live = xlive;
        float m = 0.0f;
        bool finite = true;
        if (live) {
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                finite = finite && __builtin_isfinite(v[i]);
                m = fmaxf(m, fabsf(v[i]));
            }
        }
        if (!finite) m = __builtin_inff();
#pragma unroll
        for (int off = 1; off < 32; off <<= 1) m = fmaxf(m, __shfl_xor(m, off, 64));  // the vector's 32 threads
        const int sh = split_shift(m);
        if (live) {
#pragma unroll
            for (int g = 0; g < 2; ++g) {
                half8 vh, vl;
#pragma unroll
                for (int d = 0; d < 8; ++d) {
                    const float xv = ldexpf(v[8 * g + (Tile<R>::kPermuted ? kPerm[d] : d)], sh);
                    const _Float16 th = static_cast<_Float16>(xv);
                    vh[d] = th;
                    vl[d] = static_cast<_Float16>(xv - static_cast<float>(th));
                }
                *reinterpret_cast<half8*>(&xs[0][b][c + 8 * g]) = vh;
                *reinterpret_cast<half8*>(&xs[1][b][c + 8 * g]) = vl;
            }
        }
        if (b < 8 && (threadIdx.x & 31) == 0) xmul[b] = ldexpf(1.0f, -sh);
    }
    // 3. the weights (and scales) into LDS
#pragma unroll
    for (uint32_t i = 0; i < kNU; ++i) {
        const uint32_t u = threadIdx.x + 256u * i;
        const uint32_t rr = u / kUpr, c = u - rr * kUpr;
        if (rr < TL::kRows && c * V < wdw) {
            if constexpr (V == 4) *reinterpret_cast<u32x4a*>(tl + rr * TL::kWStride + 4 * c) = wv[i];
            else tl[rr * TL::kWStride + c] = wv[i];
        }
    }
    if constexpr (kNS > 0) {
        const uint32_t sdw = Tile<R>::sdw(kc);
#pragma unroll
        for (uint32_t i = 0; i < kNS; ++i) {
            const uint32_t u = threadIdx.x + 256u * i;
            const uint32_t rr = u / kSUpr, c = u - rr * kSUpr;
            if (rr < TL::kRows && c < sdw) tl[TL::kRows * TL::kWStride + rr * TL::kSStride + c] = sv[i];
        }
    }
    __syncthreads();
    // 4. A operand rows: vector lr / 2 (the last one repeated past n_vec), part lr & 1
    const uint32_t lr = lane & 15, kg = lane >> 4;
    const _Float16* xa_row = &xs[lane & 1][(lr >> 1) < n_vec ? (lr >> 1) : n_vec - 1][0];
    constexpr int kSW = S / 4;  // slabs per wave
    f32x4 acc[kSW];
#pragma unroll
    for (int j = 0; j < kSW; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto step = [&](uint32_t bb) {
        const half8 xa = *reinterpret_cast<const half8*>(xa_row + 32 * bb + 8 * kg);
#pragma unroll
        for (int j = 0; j < kSW; ++j) {
            const uint32_t row_l = (wave + 4u * static_cast<uint32_t>(j)) * 16u + lr;
            const uint8_t* wl = reinterpret_cast<const uint8_t*>(tl + row_l * TL::kWStride);
            const uint8_t* sl = reinterpret_cast<const uint8_t*>(tl + TL::kRows * TL::kWStride + row_l * TL::kSStride);
            float sc;
            const half8 bw = Tile<R>::get(wl, sl, 0u, bb, kg, sc);
            const f32x4 z = {0.f, 0.f, 0.f, 0.f};
            const f32x4 r = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa, bw, z, 0, 0, 0);
#pragma unroll
            for (int q = 0; q < 4; ++q) acc[j][q] = __builtin_fmaf(sc, r[q], acc[j][q]);
        }
    };
    if (kc == kGemvRange) {  // a full range: four blocks' loads and products interleave
#pragma unroll 1
        for (uint32_t b0 = 0; b0 < kGemvRange / 32; b0 += 4) {
#pragma unroll
            for (uint32_t i = 0; i < 4; ++i) step(b0 + i);
        }
    } else {
        for (uint32_t bb = 0; bb < kc / 32; ++bb) step(bb);
    }
    // lane: row r0 + (wave + 4j) * 16 + lr, vectors 2kg + q (q = 0, 1) as (hi, lo) in 2q, 2q+1
#pragma unroll
    for (int j = 0; j < kSW; ++j) {
        const uint32_t row = r0 + (wave + 4u * static_cast<uint32_t>(j)) * 16u + lr;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const uint32_t jv = 2 * kg + static_cast<uint32_t>(q);
            if (jv < n_vec && row < rows)
                part[(static_cast<size_t>(blockIdx.y) * n_vec + jv) * rows + row] =
                    (acc[j][2 * q] + acc[j][2 * q + 1]) * xmul[jv];
        }
    }
}

// y[b][r] = sum over ranges s (in order) of part[s][b][r]; the loads of 8 ranges are
// in flight together, the additions keep the range order.
__global__ __launch_bounds__(256) void gemv_reduce_kernel(const float* __restrict__ part, float* __restrict__ y,
                                                          uint32_t rows, uint32_t n_vec, uint32_t n_ranges) {
    const size_t i = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x;
    const size_t n = static_cast<size_t>(n_vec) * rows;
    if (i >= n) return;
    float s = part[i];
    for (uint32_t r0 = 1; r0 < n_ranges; r0 += 8) {
        float v[8];
#pragma unroll
        for (uint32_t j = 0; j < 8; ++j)
            if (r0 + j < n_ranges) v[j] = part[static_cast<size_t>(r0 + j) * n + i];
#pragma unroll
        for (uint32_t j = 0; j < 8; ++j)
            if (r0 + j < n_ranges) s += v[j];
    }
    y[i] = s;
}

// out[t][r] = residual[t][r] + sum_j w[t][j] * part[t*k + j][r], slots in order, then
// + shared_part[t][r] (the shared expert, weight 1, last); an out-of-table id makes
// the element NaN (the id was reported by the grouping).
__global__ __launch_bounds__(256) void moe_combine_kernel(const uint32_t* __restrict__ ids, const float* __restrict__ wts,
                                                          const float* __restrict__ part,
                                                          const float* __restrict__ shared_part, const float* resid,
                                                          float* out, uint32_t k, uint32_t out_dim, uint32_t n_table) {
    const uint32_t t = blockIdx.y;
    const uint32_t r = blockIdx.x * 256 + threadIdx.x;
    if (r >= out_dim) return;
    float acc = resid ? resid[static_cast<size_t>(t) * out_dim + r] : 0.0f;
    for (uint32_t j = 0; j < k; ++j) {
        const uint32_t a = t * k + j;
        const float v = ids[a] < n_table ? part[static_cast<size_t>(a) * out_dim + r] : __builtin_nanf("");
        acc = __builtin_fmaf(wts[a], v, acc);
    }
    if (shared_part) acc += shared_part[static_cast<size_t>(t) * out_dim + r];
    out[static_cast<size_t>(t) * out_dim + r] = acc;
}

// about sixteen workgroups per CU over all slabs, at most one per member set
uint32_t grouped_gy(uint32_t rows, uint32_t max_sets, uint32_t cus) {
    const uint32_t slabs = (rows + kSlab - 1) / kSlab;
    const uint32_t want = (16 * cus + slabs - 1) / slabs;
    return want < 1 ? 1u : (want > max_sets ? max_sets : want);
}

// One grouped product launch: GATEUP over the split x rows (hidden columns) into
// act, else over the split act rows (inter columns) into part.
template <class R, bool GATEUP>
void launch_grouped_products(hipStream_t s, GroupWs gw, const _Float16* vh, const _Float16* vl, const float* vmult,
                             float* dst, uint32_t cols, uint32_t rows, uint32_t k, uint32_t n_assign, float limit,
                             bool official, uint32_t max_sets, uint32_t cus) {
    const size_t lds = (GATEUP ? 2 : 1) * 2 * 4 *
                       static_cast<size_t>(Tile<R>::lds_dw(GATEUP ? Tile<R>::kChunkGU : Tile<R>::kChunkDn));
    const dim3 grid((rows + kSlab - 1) / kSlab, grouped_gy(rows, max_sets, cus));
    if (cols % (GATEUP ? Tile<R>::kChunkGU : Tile<R>::kChunkDn) == 0)
        hipLaunchKernelGGL((moe_grouped_kernel<R, GATEUP, true>), grid, dim3(256), lds, s, gw, vh, vl, vmult, dst, cols,
                           rows, k, n_assign, limit, official ? 1u : 0u);
    else
        hipLaunchKernelGGL((moe_grouped_kernel<R, GATEUP, false>), grid, dim3(256), lds, s, gw, vh, vl, vmult, dst, cols,
                           rows, k, n_assign, limit, official ? 1u : 0u);
}

template <class R>
hipError_t launch_grouped(hipStream_t s, GroupWs gw, const _Float16* xh, const _Float16* xl, const float* xmult,
                          float* act, _Float16* ah, _Float16* al, float* amult, float* part, uint32_t n_assign,
                          uint32_t n_rows, uint32_t max_sets, uint32_t k,
                          uint32_t hidden, uint32_t inter, uint32_t out_dim, float limit, uint32_t cus) {
    launch_grouped_products<R, true>(s, gw, xh, xl, xmult, act, hidden, inter, k, n_assign, limit, false,
                                     max_sets, cus);
    hipLaunchKernelGGL(moe_split_kernel, dim3(n_rows), dim3(256), 0, s, act, inter, ah, al, amult,
                       Tile<R>::kPermuted ? 1u : 0u);
    launch_grouped_products<R, false>(s, gw, ah, al, amult, part, inter, out_dim, k, n_assign, 0.0f, false,
                                      max_sets, cus);
    return hipGetLastError();
}

}  // namespace

void launch_moe_combine(hipStream_t s, const uint32_t* ids, const float* wts, const float* part,
                        const float* shared_part, const float* resid, float* out, uint32_t n_tokens, uint32_t k,
                        uint32_t out_dim, uint32_t n_table) {
    hipLaunchKernelGGL(moe_combine_kernel, dim3((out_dim + 255) / 256, n_tokens), dim3(256), 0, s, ids, wts, part,
                       shared_part, resid, out, k, out_dim, n_table);
}

void launch_gemv_reduce(hipStream_t s, const float* part, float* y, uint32_t rows, uint32_t n_vec, uint32_t n_ranges) {
    const size_t n = static_cast<size_t>(n_vec) * rows;
    hipLaunchKernelGGL(gemv_reduce_kernel, dim3(static_cast<uint32_t>((n + 255) / 256)), dim3(256), 0, s, part, y, rows,
                       n_vec, n_ranges);
}

bool gemv_mfma_supported(int32_t format, uint64_t rows, uint64_t cols, uint64_t batch, const void* w,
                         const float* x) {
    if (batch < kGemvMfmaMinBatch || rows == 0 || rows > (1u << 24) || cols == 0 || cols > (1u << 20)) return false;
    if (reinterpret_cast<uintptr_t>(w) % 4 || reinterpret_cast<uintptr_t>(x) % 16) return false;
    if (format == OBJETA_HIP_FP4_E2M1) return cols % 128 == 0;  // the split layout
    return format >= OBJETA_HIP_Q4_0 && format <= OBJETA_HIP_IQ3_0 && cols % 64 == 0;
}

namespace {
template <class R, int S, int V>
hipError_t launch_gemv_mfma_sv(hipStream_t s, const void* w, const void* ws, const float* x, float* y, float* part,
                               uint32_t rows, uint32_t cols, uint32_t nv, uint32_t ks) {
    const uint32_t groups = (rows + 16 * S - 1) / (16 * S);
    const size_t lds = GemvTile<R, S>::lds_bytes();
    // one range: the partial sums are the result
    hipLaunchKernelGGL((gemv_mfma_kernel<R, S, V>), dim3(groups, ks), dim3(256), lds, s, w, ws, x,
                       ks > 1 ? part : y, rows, cols, nv);
    if (ks > 1) launch_gemv_reduce(s, part, y, rows, nv, ks);
    return hipGetLastError();
}

// 8 slabs (128 rows) per workgroup for Q4_0 / Q5_0 when that still gives two
// workgroups per CU, else 4; 16-byte weight units when every range is full and its
// rows 16-byte aligned. IQ3_0 and split FP4 keep 4 slabs: their 8-slab forms need
// 212 and 256 VGPRs (one or two waves per SIMD), and measured slower at 14336 x 4096
// and 8 vectors (IQ3_0 29.3 against 22.9 us, FP4 38.8 against 18.5 us), where Q4_0
// and Q5_0 gain from 8 (19.0 against 23.9, 23.0 against 33.4 us).
template <class R>
constexpr bool kGemvWideTiles = false;
template <>
constexpr bool kGemvWideTiles<QRows<kQ4>> = true;
template <>
constexpr bool kGemvWideTiles<QRows<kQ5>> = true;

template <class R>
hipError_t launch_gemv_mfma_t(hipStream_t s, const void* w, const void* ws, const float* x, float* y, float* part,
                              uint32_t rows, uint32_t cols, uint32_t nv, uint32_t ks, uint32_t cus) {
    const bool v4 = cols % kGemvRange == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0;
    if constexpr (kGemvWideTiles<R>) {
        if (static_cast<uint64_t>((rows + 127) / 128) * ks >= 2ull * cus)
            return v4 ? launch_gemv_mfma_sv<R, 8, 4>(s, w, ws, x, y, part, rows, cols, nv, ks)
                      : launch_gemv_mfma_sv<R, 8, 1>(s, w, ws, x, y, part, rows, cols, nv, ks);
    }
    return v4 ? launch_gemv_mfma_sv<R, 4, 4>(s, w, ws, x, y, part, rows, cols, nv, ks)
              : launch_gemv_mfma_sv<R, 4, 1>(s, w, ws, x, y, part, rows, cols, nv, ks);
}
}  // namespace

size_t gemv_passes_bytes(uint64_t rows, uint64_t cols, uint64_t batch) {
    const uint64_t ks = (cols + kGemvRange - 1) / kGemvRange;
    return ks > 1 ? 4 * ks * (batch < 8 ? batch : 8) * rows : 0;
}

int32_t launch_gemv_mfma(objeta_hip_context* ctx, hipStream_t s, int32_t format, const void* w, const void* ws,
                         const float* x, float* y, uint64_t rows, uint64_t cols, uint64_t batch) {
    const char* action = "launch batched GEMV (MFMA)";
    if (!gemv_mfma_supported(format, rows, cols, batch, w, x))
        OBJ_FAIL(kUnsupported, action, "shape, batch or alignment outside the MFMA GEMV");
    // (under capture without its workspace, the passes below, which need less or none)
    if (gemv_wide_supported(format, rows, cols, batch) &&
        workspace_ready(ctx, s, kWsGemv, gemv_wide_bytes(ctx, format, rows, cols, batch)))
        return launch_gemv_wide(ctx, s, format, w, ws, x, y, rows, cols, batch);
    const uint32_t R = static_cast<uint32_t>(rows), K = static_cast<uint32_t>(cols);
    const uint32_t ks = (K + kGemvRange - 1) / kGemvRange;  // column ranges
    const uint32_t cus = ctx->info.compute_units > 0 ? static_cast<uint32_t>(ctx->info.compute_units) : 256u;
    float* part = nullptr;
    if (ks > 1) {
        void* wsp = nullptr;
        OBJ_TRY(ensure_workspace(ctx, s, kWsGemv, gemv_passes_bytes(rows, cols, batch), &wsp));
        part = static_cast<float*>(wsp);
    }
    for (uint64_t done = 0; done < batch; done += 8) {
        const uint32_t nv = static_cast<uint32_t>(batch - done < 8 ? batch - done : 8);
        const float* xb = x + done * cols;
        float* yb = y + done * rows;
        hipError_t e;
        switch (format) {
            case OBJETA_HIP_Q4_0: e = launch_gemv_mfma_t<QRows<kQ4>>(s, w, nullptr, xb, yb, part, R, K, nv, ks, cus); break;
            case OBJETA_HIP_Q5_0: e = launch_gemv_mfma_t<QRows<kQ5>>(s, w, nullptr, xb, yb, part, R, K, nv, ks, cus); break;
            case OBJETA_HIP_IQ3_0: e = launch_gemv_mfma_t<QRows<kIQ3>>(s, w, nullptr, xb, yb, part, R, K, nv, ks, cus); break;
            default: e = launch_gemv_mfma_t<Fp4Rows>(s, w, ws, xb, yb, part, R, K, nv, ks, cus); break;
        }
        if (e != hipSuccess) OBJ_FAIL(kDriver, action, hipGetErrorString(e));
    }
    return 0;
}

// Whether a batch has so few assignments (token, slot; the shared expert is one more slot)
// that the sets of eight are the faster form. The wide products make a work item of 64
// weight rows per expert and walk its columns in one chain with one LDS buffer; with fewer
// work items than the CUs take at once, that chain is the time. A set of eight takes 16 rows
// of each matrix with two buffers: more workgroups per expert, until the weights' bytes are
// the time or experts have more than eight of the tokens (their weights are read again).
// IQ3_0, the dearest to decode, and split FP4 turn earlier. us per layer, wide products /
// sets of eight (64 experts, 2048 x 768: 128; Zipf popularity), below | past the line:
//   Q4_0 4096 x 1536  top-1, 12 tokens 61 / 47, top-2, 24 85 / 83 | top-4, 24 120 / 127
//   Q4_0 7168 x 2048  top-1, 9 tokens 92 / 74, top-4, 10 177 / 173 | top-4, 12 187 / 188
//   Q5_0 2048 x 1408  top-1, 12 tokens 49 / 36, top-2, 32 60 / 56 | top-8, 14 84 / 85
//   IQ3_0 2048 x 768  top-1, 12 tokens 38 / 35, top-2, 16 41 / 40 | top-4, 12 45 / 46
//   FP4 7168 x 2048   top-1, 2 tokens 80 / 51, top-2, 8 115 / 109 | top-2, 10 121 / 122
//   FP4 4608 x 1664   top-2, 5 tokens 64 / 56, top-1, 32 92 / 89 | top-4, 12 108 / 114
//   FP4 4096 x 1408   top-2, 8 tokens 63 / 54, top-8, 4 89 / 80 | top-8, 8 106 / 108
// The largest losses near the line over 620 such layers: FP4 7168 x 2048 top-8, 2 tokens 122
// / 132 below, 4096 x 1408 top-4, 12 tokens 93 / 87 past it.
bool few_assignments(int32_t format, uint64_t n_table, uint64_t n_tokens, uint64_t k, bool shared, uint64_t hidden,
                     uint64_t inter, uint64_t out_dim) {
    if (k == 0 || k > 32 || n_table == 0 || n_table > kGMaxTable || n_tokens > kGMaxAssign) return false;
    if (hidden > (1u << 20) || inter > (1u << 20) || out_dim > (1u << 20)) return false;
    // one matrix's weights over all assignments (the limits also keep its offsets in 32 bits)
    const uint64_t a = n_tokens * (k + (shared ? 1 : 0)), weights = a * inter * (hidden > out_dim ? hidden : out_dim);
    switch (format) {
        case OBJETA_HIP_Q4_0:
        case OBJETA_HIP_Q5_0: return a <= 72 && weights <= 640u << 20;
        case OBJETA_HIP_IQ3_0: return a <= 40 && weights <= 96u << 20;
        default: return a <= 40 && weights <= 240u << 20;
    }
}

bool grouped_supported(int32_t format, uint64_t n_table, uint64_t n_tokens, uint64_t k, uint64_t hidden,
                       uint64_t inter, uint64_t out_dim) {
    if (format < OBJETA_HIP_Q4_0 || format > OBJETA_HIP_FP4_E2M1) return false;
    if (wide_supported(format, n_table, n_tokens, k, hidden, inter, out_dim)) return true;
    if (k == 0 || k > 32 || n_table == 0 || n_table > kGMaxTable || n_tokens * k > kGMaxAssign) return false;
    if (hidden == 0 || inter == 0 || hidden % 64 || inter % 64 || hidden > (1u << 20) || inter > (1u << 20) ||
        out_dim > (1u << 20))
        return false;
    // split FP4 runs on the sets of eight for few assignments alone, which are wide_supported
    return format != OBJETA_HIP_FP4_E2M1 && matrices_fit(format, false, hidden, inter, out_dim);
}

namespace {
// The layout for T tokens; the pointers of w are set when base is.
size_t grouped_layout(uint64_t T, uint64_t k, uint64_t n_table, bool shared, uint64_t H, uint64_t I, uint64_t O,
                      bool official, char* base, GroupedWs* w) {
    const uint64_t A = T * k, NR = A + (shared ? T : 0), n8 = shared ? (T + 7) / 8 : 0, n16 = shared ? (T + 15) / 16 : 0;
    auto larger = [](uint64_t a, uint64_t b) { return a > b ? a : b; };
    auto whole = [](uint64_t n) { return (n + 7) & ~uint64_t(7); };  // rounds of the eight XCDs
    size_t off = 0;
    auto take = [&](size_t bytes) {
        char* const at = base ? base + off : nullptr;
        off += (bytes + 255) & ~size_t(255);
        return at;
    };
    GroupedWs g;
    g.hdr = reinterpret_cast<uint32_t*>(take(16));
    g.sets = take(larger(sizeof(SetRec) * (A + n8), kWideSetBytes * whole((A < n_table ? A : n_table) + A / 16 + n16)));
    g.shared_sets = take(larger(sizeof(SetRec) * n8, kWideSetBytes * whole(n16)));
    g.xd = reinterpret_cast<float*>(take(official ? 4 * T * H : 0));
    g.xmult = reinterpret_cast<float*>(take(4 * T));
    g.amult = reinterpret_cast<float*>(take(4 * NR));
    g.xh = reinterpret_cast<_Float16*>(take(2 * T * H));
    g.xl = reinterpret_cast<_Float16*>(take(2 * T * H));
    g.act = reinterpret_cast<float*>(take(4 * NR * I));
    g.ah = reinterpret_cast<_Float16*>(take(2 * NR * I));
    g.al = reinterpret_cast<_Float16*>(take(2 * NR * I));
    g.part = reinterpret_cast<float*>(take(4 * NR * O));
    if (w) *w = g;
    return off;
}
}  // namespace

int32_t grouped_workspace(objeta_hip_context* ctx, hipStream_t s, uint64_t n_tokens, uint64_t k, uint64_t n_table,
                          bool shared, uint64_t hidden, uint64_t inter, uint64_t out_dim, bool official, GroupedWs& w) {
    void* p = nullptr;
    OBJ_TRY(ensure_workspace(ctx, s, kWsGrouped,
                             grouped_layout(n_tokens, k, n_table, shared, hidden, inter, out_dim, official, nullptr, nullptr), &p));
    (void)grouped_layout(n_tokens, k, n_table, shared, hidden, inter, out_dim, official, static_cast<char*>(p), &w);
    return 0;
}

bool grouped_ready(objeta_hip_context* ctx, hipStream_t s, int32_t format, uint64_t n_table, uint64_t n_tokens, uint64_t k,
                   bool shared, uint64_t hidden, uint64_t inter, uint64_t out_dim, bool official) {
    uint64_t t = n_tokens;
    if (wide_supported(format, n_table, n_tokens, k, hidden, inter, out_dim) && t > wide_tokens(k, hidden, inter))
        t = wide_tokens(k, hidden, inter);
    return workspace_ready(ctx, s, kWsGrouped,
                           grouped_layout(t, k, n_table, shared, hidden, inter, out_dim, official, nullptr, nullptr));
}

bool grouped_preferred(int32_t format, uint64_t n_tokens, uint64_t k, bool shared, uint64_t hidden, uint64_t inter,
                       uint64_t out_dim) {
    if (n_tokens >= kGroupedMinTokens) return true;
    if (n_tokens < 2) return false;
    // bytes per 32 weights of each format
    const uint64_t per32 = format == OBJETA_HIP_Q4_0 ? 18 : format == OBJETA_HIP_Q5_0 ? 22
                         : format == OBJETA_HIP_IQ3_0 ? 14 : 17;
    const uint64_t bytes = (2 * inter * hidden + out_dim * inter) / 32 * per32;
    if (bytes >= kGroupedLargeExpertBytes) return true;
    if (k > 32) return false;
    const uint64_t groups = hidden / 64;  // of 64 columns, one to a lane
    if (inter <= 1024 && groups >= 32 && (groups & (groups - 1)) == 0) {
        const bool dear = format == OBJETA_HIP_Q5_0 || format == OBJETA_HIP_IQ3_0;
        if (groups > 64) return false;
        if (groups == 64) {
            const uint64_t limit = dear ? kGroupedReadBytesDear4096 : shared ? kGroupedReadBytesShared4096 : kGroupedReadBytes4096;
            return n_tokens * (k + (shared ? 1 : 0)) * bytes >= limit;
        }
        if (!dear && !shared) return n_tokens * k * bytes >= kGroupedReadBytes2048;
    }
    return n_tokens * k * bytes >= kGroupedReadBytes;
}

int32_t launch_moe_grouped(objeta_hip_context* ctx, int32_t format, hipStream_t s, const objeta_hip_expert_ptrs* table,
                           uint64_t n_table, const objeta_hip_expert_ptrs* shared, const uint32_t* ids, const float* wts,
                           uint64_t n_tokens, uint64_t k, const float* x, const float* resid, float* out, uint64_t hidden, uint64_t inter,
                           uint64_t out_dim, float limit) {
    const char* action = "launch grouped-token MoE";
    if (format < OBJETA_HIP_Q4_0 || format > OBJETA_HIP_FP4_E2M1)
        OBJ_FAIL(kInvalidInput, action, strf("unknown format %d", format));
    if (n_tokens == 0 || out_dim == 0) return 0;
    const bool few = few_assignments(format, n_table, n_tokens, k, shared != nullptr, hidden, inter, out_dim);
    if (!few && wide_supported(format, n_table, n_tokens, k, hidden, inter, out_dim))
        return launch_moe_wide(ctx, format, s, table, n_table, shared, ids, wts, n_tokens, k, x, resid, out, hidden, inter,
                               out_dim, limit);
    if (k == 0 || k > 32) OBJ_FAIL(kInvalidInput, action, "k must be in 1..=32");
    if (n_table == 0 || n_table > kGMaxTable)
        OBJ_FAIL(kUnsupported, action, strf("the grouped path takes up to %u experts", kGMaxTable));
    if (n_tokens * k > kGMaxAssign)
        OBJ_FAIL(kUnsupported, action, strf("the grouped path takes up to %u (token, slot) assignments", kGMaxAssign));
    if (hidden == 0 || inter == 0 || hidden % 64 || inter % 64 || hidden > (1u << 20) || inter > (1u << 20) ||
        out_dim > (1u << 20))
        OBJ_FAIL(kUnsupported, action, "hidden and intermediate must be non-zero multiples of 64 (<= 2^20)");
    if (format == OBJETA_HIP_FP4_E2M1 && (hidden % 128 || inter % 128))
        OBJ_FAIL(kUnsupported, action, "the grouped path takes split-FP4 experts with hidden and intermediate % 128 == 0");
    if (!matrices_fit(format, false, hidden, inter, out_dim)) OBJ_FAIL(kUnsupported, action, "matrices above 2^31 bytes");
    if (!table || !ids || !wts || !x || !out) OBJ_FAIL(kInvalidInput, action, "NULL device pointer");
    if (reinterpret_cast<uintptr_t>(x) % 16) OBJ_FAIL(kInvalidInput, action, "x must be 16-byte aligned");
    const uint32_t A = static_cast<uint32_t>(n_tokens * k), T = static_cast<uint32_t>(n_tokens);
    const uint32_t NR = A + (shared ? T : 0);                  // act rows: routed, then shared
    const uint32_t NS = A + (shared ? (T + 7) / 8 : 0);        // member sets at most
    const uint32_t H = static_cast<uint32_t>(hidden), I = static_cast<uint32_t>(inter), O = static_cast<uint32_t>(out_dim);
    GroupedWs w;
    OBJ_TRY(grouped_workspace(ctx, s, T, k, n_table, shared != nullptr, hidden, inter, out_dim, false, w));
    const GroupWs gw{w.hdr, static_cast<SetRec*>(w.sets)};
    float *const amult = w.amult, *const xmult = w.xmult, *const act = w.act, *const part = w.part;
    _Float16 *const xh = w.xh, *const xl = w.xl, *const ah = w.ah, *const al = w.al;
    uint32_t* err = ctx->err_word;
    const uint32_t cus = ctx->info.compute_units > 0 ? static_cast<uint32_t>(ctx->info.compute_units) : 256u;
    // the split order follows the weights' order (element order for FP4)
    const bool perm = format == OBJETA_HIP_FP4_E2M1 ? Tile<Fp4Rows>::kPermuted : Tile<QRows<kQ4>>::kPermuted;
    hipLaunchKernelGGL(moe_prepare_kernel, dim3(1 + T), dim3(256), 0, s, ids, A, static_cast<uint32_t>(n_table), table,
                       shared, T, gw, GroupWs{nullptr, nullptr}, err, x, H, xh, xl, xmult, perm ? 1u : 0u);
    hipError_t e;
    const uint32_t kk = static_cast<uint32_t>(k);
    switch (format) {
        case OBJETA_HIP_Q4_0:
            e = launch_grouped<QRows<kQ4>>(s, gw, xh, xl, xmult, act, ah, al, amult, part, A, NR, NS, kk, H,
                                           I, O, limit, cus);
            break;
        case OBJETA_HIP_Q5_0:
            e = launch_grouped<QRows<kQ5>>(s, gw, xh, xl, xmult, act, ah, al, amult, part, A, NR, NS, kk, H,
                                           I, O, limit, cus);
            break;
        case OBJETA_HIP_IQ3_0:
            e = launch_grouped<QRows<kIQ3>>(s, gw, xh, xl, xmult, act, ah, al, amult, part, A, NR, NS, kk,
                                            H, I, O, limit, cus);
            break;
        default:
            e = launch_grouped<Fp4Rows>(s, gw, xh, xl, xmult, act, ah, al, amult, part, A, NR, NS, kk, H, I,
                                        O, limit, cus);
            break;
    }
    if (e == hipSuccess) {
        launch_moe_combine(s, ids, wts, part, shared ? part + static_cast<size_t>(A) * O : nullptr, resid, out, T, kk, O,
                           static_cast<uint32_t>(n_table));
        e = hipGetLastError();
    }
    if (e != hipSuccess) OBJ_FAIL(kDriver, action, hipGetErrorString(e));
    return 0;
}

// Few assignments on large matrices, as for the plain layer, but the line is set by the FP8
// shared expert: its rows are the longest, and on the wide products its one set walks them in
// inter / 32 workgroups. us, wide / here, with the shared expert, below | past the line: 7168 x
// 2048 top-1, 4 tokens 115 / 92, 14, 117 / 113, top-2, 6, 118 / 113 | 8, 117 / 122, top-4, 3,
// 122 / 124; 4608 x 1664 top-1, 8, 87 / 79 | top-2, 10, 93 / 97; 4096 x 1408 top-1, 6, 72 / 66 |
// 20, 73 / 78; 7168 x 768 top-1, 8 | 86 / 88; 2048 x 2048 top-2, 6 | 53 / 55.
bool official_few(uint64_t n_table, uint64_t n_tokens, uint64_t k, uint64_t hidden, uint64_t inter, uint64_t out_dim) {
    if (k == 0 || k > 2 || n_table == 0 || n_table > kGMaxTable || n_tokens > 14) return false;
    if (hidden > (1u << 20) || inter > (1u << 20) || out_dim > (1u << 20)) return false;
    return n_tokens * k <= 14 && inter > 1024 && hidden * inter >= (uint64_t(5) << 20);
}

// The official layer (launch_moe_official_grouped) on the sets of eight: the FP8 shared
// expert's sets apart, in a launch of their own per phase.
int32_t launch_moe_official_sets(objeta_hip_context* ctx, hipStream_t s, const objeta_hip_expert_ptrs* table,
                                 uint64_t n_table, const objeta_hip_expert_ptrs* shared, const uint32_t* ids,
                                 const float* wts, uint64_t n_tokens, uint64_t k, const float* x, float* out,
                                 uint64_t hidden, uint64_t inter, uint64_t out_dim, float limit,
                                 uint8_t* inter_values, uint8_t* inter_scales) {
    const char* action = "launch official FP4 MoE (sets of eight)";
    const uint32_t T = static_cast<uint32_t>(n_tokens), A = static_cast<uint32_t>(n_tokens * k);
    const uint32_t NR = A + (shared ? T : 0);       // act rows: routed, then shared
    const uint32_t NSS = shared ? (T + 7) / 8 : 0;  // shared member sets
    const uint32_t H = static_cast<uint32_t>(hidden), I = static_cast<uint32_t>(inter), O = static_cast<uint32_t>(out_dim);
    GroupedWs w;
    OBJ_TRY(grouped_workspace(ctx, s, T, k, n_table, shared != nullptr, hidden, inter, out_dim, true, w));
    const GroupWs gw{w.hdr, static_cast<SetRec*>(w.sets)}, gws{w.hdr + 2, static_cast<SetRec*>(w.shared_sets)};
    float *const xd = w.xd, *const xmult = w.xmult, *const amult = w.amult, *const act = w.act, *const part = w.part;
    _Float16 *const xh = w.xh, *const xl = w.xl, *const ah = w.ah, *const al = w.al;
    const uint32_t cus = ctx->info.compute_units > 0 ? static_cast<uint32_t>(ctx->info.compute_units) : 256u;
    const uint32_t kk = static_cast<uint32_t>(k), perm = Tile<Fp4Rows>::kPermuted ? 1u : 0u;
    OBJ_TRY(launch_act_quant(s, x, T, H, nullptr, nullptr, xd));
    hipLaunchKernelGGL(moe_prepare_kernel, dim3(1 + T), dim3(256), 0, s, ids, A, static_cast<uint32_t>(n_table), table,
                       shared, T, gw, shared ? gws : GroupWs{nullptr, nullptr}, ctx->err_word, xd, H, xh, xl, xmult, perm);
    launch_grouped_products<Fp4Rows, true>(s, gw, xh, xl, xmult, act, H, I, kk, A, limit, true, A, cus);
    if (shared) launch_grouped_products<Fp8Rows, true>(s, gws, xh, xl, xmult, act, H, I, kk, A, limit, true, NSS, cus);
    OBJ_HIP(hipGetLastError(), action);
    OBJ_TRY(launch_act_quant(s, act, NR, I, inter_values, inter_scales, act));
    hipLaunchKernelGGL(moe_split_kernel, dim3(NR), dim3(256), 0, s, act, I, ah, al, amult, perm);
    launch_grouped_products<Fp4Rows, false>(s, gw, ah, al, amult, part, I, O, kk, A, 0.0f, false, A, cus);
    if (shared) launch_grouped_products<Fp8Rows, false>(s, gws, ah, al, amult, part, I, O, kk, A, 0.0f, false, NSS, cus);
    launch_moe_combine(s, ids, wts, part, shared ? part + static_cast<size_t>(A) * O : nullptr, nullptr, out, T, kk, O,
                       static_cast<uint32_t>(n_table));
    OBJ_HIP(hipGetLastError(), action);
    return 0;
}

}  // namespace objeta

using namespace objeta;

extern "C" int32_t objeta_hip_moe_grouped_device(objeta_hip_context* ctx, int32_t format, objeta_hip_stream stream,
                                                 const objeta_hip_expert_ptrs* d_table, uint64_t n_table,
                                                 const uint32_t* d_ids, const float* d_weights, uint64_t n_tokens,
                                                 uint64_t k, const float* d_x, const float* d_residual, float* d_out,
                                                 uint64_t hidden, uint64_t intermediate, uint64_t out_dim,
                                                 float swiglu_limit) {
    OBJ_GUARD_BEGIN
    OBJ_TRY(check_ctx(ctx, "moe_grouped_device"));
    OBJ_HIP(hipSetDevice(ctx->device), "hipSetDevice");
    if (format >= OBJETA_HIP_Q4_0 && format <= OBJETA_HIP_FP4_E2M1 && n_tokens && out_dim && k && k <= 32 && n_table &&
        n_table <= kGMaxTable && n_tokens * k > kGMaxAssign)
        OBJ_FAIL(kUnsupported, "launch grouped-token MoE",
                 strf("the grouped path takes up to %u (token, slot) assignments", kGMaxAssign));
    return launch_moe_grouped(ctx, format, resolve_stream(ctx, stream), d_table, n_table, nullptr, d_ids, d_weights,
                              n_tokens, k, d_x, d_residual, d_out, hidden, intermediate, out_dim, swiglu_limit);
    OBJ_GUARD_END
}

// Varlen paged attention for gfx950: one code path for decode, chunked
// prefill and the (k+1)-query speculative verify.
//
// Work decomposition. A "column" is one (query row, query head) pair; the G
// query heads that share a KV head are adjacent columns, so a decode row of a
// GQA group-5 model is 5 columns and a 5-token verify row of a group-3 model is
// 15. One wave owns a work item = (sequence, kv head, up to NT tiles of 16
// columns, a range of 16-key tiles), reads every K/V tile of that range exactly
// once and shares it across all of its columns.
//
// Per 16-key tile the wave computes S^T = K Q^T with MFMA (A = K rows straight
// from the pool, B = the Q fragment kept in registers), applies the per-column
// causal rule key <= position(row), runs the online softmax with the column
// max reduced across the four 16-lane groups by xor shuffles, and accumulates
// O^T = V^T P^T with a second MFMA whose B operand is the exponentiated S^T
// tile exactly as the first MFMA left it in registers. V arrives with
// fully coalesced 16-token x 16-byte row loads and is transposed into the MFMA
// A layout with byte permutes. 16-bit prefill runs in workgroups that share
// each K/V row through LDS instead (attn_wide_body).
//
// Long contexts are split into key partitions (the plan decides); each leaves
// its running maximum and sum in fp32 and its normalised output in the launch's
// type (or in fp32, see the split-K merge), and a merge kernel combines them
// with the log-sum-exp rule.
#include <algorithm>
#include <array>
#include <atomic>
#include <climits>
#include <cmath>
#include <mutex>
#include <type_traits>
#include <vector>

#include "mf_common.h"

#ifndef MF_MAX_ITEM_TILES
#define MF_MAX_ITEM_TILES 128
#endif
namespace mf {
namespace {

typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef __attribute__((ext_vector_type(4))) short i16x4;
typedef __attribute__((ext_vector_type(4))) _Float16 f16x4;

constexpr int kWaves = 4;  // waves per workgroup; each wave runs its own item
constexpr int kMaxItemTiles = MF_MAX_ITEM_TILES;  // key tiles per work item (two block-table entries per lane)
#ifndef MF_NARROW_ITEMS
#define MF_NARROW_ITEMS 4096  // planner: target item count that sets the narrow key partition
#endif
// Wave priority (s_setprio) of the workgroup-shared wide loop. In a mixed
// launch a CU holds single-tile (decode) waves beside the wide (prefill) ones;
// at equal priority the decode waves' issue slowed the wide workgroups sharing
// their CU by about 40% (per-workgroup timestamps on the C2 step: 31.4 against
// 22.0 us median life), and the CUs holding a decode workgroup finished last.
// Raised, the wide waves issue first and the decode waves take the slots they
// leave while they wait on memory. Measured on the C2 engine layer: 53.7 us at
// equal priority, 49.3-49.8 us at 1, 49.4-49.8 at 2.
#ifndef MF_WIDE_PRIO
#define MF_WIDE_PRIO 1
#endif
// XCD-local order of the wide workgroups (1). The dispatcher sends
// workgroup b of a launch to XCD b mod 8, so the
// consecutive wide workgroups of one key range (the column groups of one
// sequence, kv head and key partition, which read the same K/V tiles) land on
// eight XCDs whose L2s each fetch the tiles. The planner instead deals whole
// ranges to eight queues (least causal work first) and interleaves them, so
// workgroup 8k + x comes from queue x and a range stays on one XCD; each
// queue runs its workgroups most causal work first. Measured on the C2
// prefill items alone: 38.2-38.8 us -> 35.1-35.5 us between events, PMC
// FETCH 74 MB -> 24 MB (1.4x the K/V and query bytes). In a mixed launch the
// wide workgroups follow the single-tile ones, which only rotates the XCDs
// (a range still shares one). There, at 32-tile wide partitions, the order
// was slower (C2 engine layer 49.2 -> 50.2 us); at 64-tile equal-stride
// partitions it was faster: 45.71-45.75 against 45.85-45.94 us, and the mixed
// plan's prefill items alone 34.7-34.9 against 39.6-39.8 us. Mixed plans now
// cut each column quad on its own (quad partitions, in the planner) and keep
// a (sequence, kv head)'s workgroups on one XCD.
#ifndef MF_WIDE_XCD
#define MF_WIDE_XCD 1
#endif
#ifndef MF_WIDE_ITEMS
#define MF_WIDE_ITEMS 4096  // planner: most wide items before partitions grow
#endif
constexpr float kLazyLog2 = 8.f;  // running-max slack of the online softmax (log2 units)
// Running maximum before any key is seen: finite, so exponent arguments never
// need a -inf guard; 2^(kMinM - x) is 0 for every score x.
constexpr float kMinM = -1e30f;

// 16-column tiles one wave carries for multi-tile (prefill / wide verify)
// items.
__host__ __device__ constexpr int wide_tiles(int dt, int dp) {
    // 16-bit: the 32 columns of one MFMA block (attn_wide_body)
    return dt == MF_F32 ? (dp >= 128 ? 2 : 4) : (dp >= 256 ? 1 : 2);
}

struct AttnArgs {
    const char* q;
    int64_t q_sr, q_sh;
    char* out;
    int64_t o_sr, o_sh;
    const char* k_pool;
    const char* v_pool;
    int64_t p_sb, p_ss, p_sh;
    int block_size;
    const int32_t* block_tables;
    int64_t bt_stride;
    const int32_t* cu_seqlens;
    const int32_t* kv_lens;
    const int64_t* positions;
    const int32_t* row_map;
    const int32_t* pool_lens;
    const char* new_k;
    const char* new_v;
    int64_t n_sr, n_sh;
    int G;
    int head_dim;
    float scale_log2;    // |scale| * log2(e), > 0
    float inv_scale_log2;
    uint32_t q_sign;     // xor applied to every Q word: flips the sign for a negative scale
    const int32_t* items;
    int num_items;
    const int32_t* dev_count;  // when set, the live item / merge count (the grid is a capacity)
    float* partials;
    int part_dstride;  // floats per column of a partial slot's output block
    const int32_t* merges;  // plan merge records (fused split-K merge)
    int32_t* counters;      // per-group arrival counters; null = separate merge kernel
    // Written-in-flight launch (mf_paged_attention_kv_write; the kernels'
    // TAIL instances): a sequence's keys at or above kv_len - rows are its own
    // new rows, read from new_k/new_v (row cu_seqlens[s] + key - (kv_len -
    // rows)), and the launch's first w_blocks workgroups copy new rows
    // [0, w_rows) into the pool through w_slots (a slot < 0 or >= w_num_slots
    // is skipped). No item reads a slot that this launch writes, so nothing
    // waits on the copy.
    int num_kv_heads;
    const int64_t* w_slots;
    int w_rows;
    int w_blocks;
    int64_t w_num_slots;
};

// The copy of a written-in-flight launch: workgroup `wblock` of the leading
// w_blocks. Every new row's K and V, head by head, go to the pool slot of
// w_slots in 16-byte pieces: consecutive lanes take consecutive pieces of one
// row (its heads are adjacent), so loads and stores coalesce.
template <int DT>
__device__ __forceinline__ void write_new_rows(const AttnArgs& a, int wblock) {
    constexpr int ES = DT == MF_F32 ? 4 : 2;
    const int cpr = a.head_dim * ES / 16;  // 16-byte pieces of one head's row
    const int per_row = 2 * a.num_kv_heads * cpr;
    const int total = a.w_rows * per_row;
    for (int u = wblock * 256 + (int)threadIdx.x; u < total; u += a.w_blocks * 256) {
        const int row = u / per_row;
        int rest = u - row * per_row;
        const int isv = rest >= a.num_kv_heads * cpr;
        rest -= isv * a.num_kv_heads * cpr;
        const int head = rest / cpr;
        const int piece = rest - head * cpr;
        const int64_t slot = a.w_slots[row];
        if (slot < 0 || slot >= a.w_num_slots) continue;
        const int64_t blk = slot / a.block_size;
        const int64_t off = slot - blk * a.block_size;
        const char* src = (isv ? a.new_v : a.new_k) + ((int64_t)row * a.n_sr + (int64_t)head * a.n_sh) * ES + piece * 16;
        char* dst = const_cast<char*>(isv ? a.v_pool : a.k_pool) +
                    (blk * a.p_sb + off * a.p_ss + (int64_t)head * a.p_sh) * ES + piece * 16;
        *(uint4*)dst = *(const uint4*)src;
    }
}

// ------------------------------------------------------------- MFMA wrappers
// S^T tile: 16 keys x 16 columns, contraction over one 16-byte chunk of
// head_dim per lane (8 x 16-bit or 4 x fp32 elements).
template <int DT>
__device__ __forceinline__ f32x4 mfma_qk(uint4 a, uint4 b, f32x4 c) {
    if constexpr (DT == MF_BF16) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                       __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    } else if constexpr (DT == MF_F16) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                      __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    } else {
        c = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a.x), __uint_as_float(b.x), c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a.y), __uint_as_float(b.y), c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a.z), __uint_as_float(b.z), c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a.w), __uint_as_float(b.w), c, 0, 0, 0);
        return c;
    }
}

// O^T tile: 16 head_dim rows x 16 columns, contraction over 16 keys
// (4 per lane) for 16-bit types.
template <int DT>
__device__ __forceinline__ f32x4 mfma_pv16(uint2 a, uint2 b, f32x4 c) {
    if constexpr (DT == MF_BF16) {
        return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(i16x4, a),
                                                         __builtin_bit_cast(i16x4, b), c, 0, 0, 0);
    } else {
        return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(f16x4, a),
                                                     __builtin_bit_cast(f16x4, b), c, 0, 0, 0);
    }
}

// ---------------------------------------------------------- memory helpers

template <int N>
__device__ __forceinline__ void ld_words(const char* p, uint32_t* w) {
    if constexpr (N == 4) {
        w[0] = *(const uint32_t*)p;
    } else if constexpr (N == 8) {
        const uint2 v = *(const uint2*)p;
        w[0] = v.x; w[1] = v.y;
    } else {
        static_assert(N % 16 == 0, "chunk");
#pragma unroll
        for (int k = 0; k < N / 16; ++k) {
            const uint4 v = *(const uint4*)(p + 16 * k);
            w[4 * k] = v.x; w[4 * k + 1] = v.y; w[4 * k + 2] = v.z; w[4 * k + 3] = v.w;
        }
    }
}

// The same loads marked non-temporal (streamed, not kept in cache): pool
// tiles of single-column-tile items are read by exactly one wave.
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ uint4 ld_nt16(const char* p) {
    const u32x4 v = __builtin_nontemporal_load((const u32x4*)p);
    return make_uint4(v.x, v.y, v.z, v.w);
}
// 16 bytes per lane from global memory straight into LDS (gfx950's
// global_load_lds_dwordx4): lane i's bytes land at lds_addr + 16 i, lds_addr
// being the same for the whole wave. Written as inline assembly because the
// builtin makes the compiler wait for the transfer before every later LDS
// read; the caller waits for it (vmcnt) before the barrier that publishes it.
// The LDS address is bound to m0 by the operand constraint, so the compiler
// writes m0 itself and knows what it holds (a clobber of the reserved m0
// would not be honoured); the s_nop gives the write its one wait state before
// the load reads it.
__device__ __forceinline__ void ld_lds16(const void* gsrc, uint32_t lds_addr) {
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"{m0}"(lds_addr), "v"(gsrc) : "memory");
}

template <int N>
__device__ __forceinline__ void ld_words_nt(const char* p, uint32_t* w) {
    if constexpr (N == 4) {
        w[0] = __builtin_nontemporal_load((const uint32_t*)p);
    } else if constexpr (N == 8) {
        const u32x2 v = __builtin_nontemporal_load((const u32x2*)p);
        w[0] = v.x; w[1] = v.y;
    } else {
        static_assert(N % 16 == 0, "chunk");
#pragma unroll
        for (int k = 0; k < N / 16; ++k) {
            const uint4 v = ld_nt16(p + 16 * k);
            w[4 * k] = v.x; w[4 * k + 1] = v.y; w[4 * k + 2] = v.z; w[4 * k + 3] = v.w;
        }
    }
}

template <int N>
__device__ __forceinline__ void st_words(char* p, const uint32_t* w) {
    if constexpr (N == 4) {
        *(uint32_t*)p = w[0];
    } else if constexpr (N == 8) {
        *(uint2*)p = make_uint2(w[0], w[1]);
    } else {
        static_assert(N % 16 == 0, "chunk");
#pragma unroll
        for (int k = 0; k < N / 16; ++k)
            *(uint4*)(p + 16 * k) = make_uint4(w[4 * k], w[4 * k + 1], w[4 * k + 2], w[4 * k + 3]);
    }
}

// Writes NE contiguous output elements (value e is vals[e]) in dtype DT.
template <int DT, int NE>
__device__ __forceinline__ void store_elems(char* p, const float* vals) {
    if constexpr (DT == MF_F32) {
        uint32_t w[NE];
#pragma unroll
        for (int e = 0; e < NE; ++e) w[e] = __float_as_uint(vals[e]);
        st_words<NE * 4>(p, w);
    } else {
        uint32_t w[NE / 2];
#pragma unroll
        for (int e = 0; e < NE / 2; ++e)
            w[e] = f32_to_bits<DT>(vals[2 * e]) | (f32_to_bits<DT>(vals[2 * e + 1]) << 16);
        st_words<NE * 2>(p, w);
    }
}

// Writes the lane's contiguous chunk of 4*VCH output elements.
template <int DT, int VCH>
__device__ __forceinline__ void store_out_chunk(char* p, const float* vals) {
    store_elems<DT, 4 * VCH>(p, vals);
}

// ------------------------------------------------------------- split-K merge
// Partials of one 16-column tile (merge record `mg`) live in slots
// slot0 + p*sstride, p < np. A slot holds, per column, the partition's
// normalised output o_p / l_p in the launch's element type (column c at
// element c*part_dstride), then 16 running maxima m_p and 16 sums l_p (fp32,
// at float 16*part_dstride). The merged output is
// sum_p w_p l_p (o_p / l_p) / sum_p w_p l_p with w_p = 2^(m_p - max_p m_p).
// A normalised output is a convex combination of V rows, so it keeps the
// output type's range; 16-bit partials halve the bytes written and merged
// against fp32 ones, for one more rounding to that type.
// Records and items flagged MF_PLAN_FP32_PARTIALS hold the outputs in fp32
// instead (the slot has the room): a device's decode plan cuts ranges that the
// general plan runs as one cooperative unit, whose waves combine in fp32, and the
// cut must not round what the whole unit does not. 16-bit launches of 256-byte
// rows and more only, as that rule.
template <int DT, int DP>
constexpr bool has_fp32_partials() { return DT != MF_F32 && DP >= 128; }
template <int DT>
__device__ __forceinline__ char* partial_out(const AttnArgs& a, int64_t slot, int col, int elem) {
    constexpr int ES = DT == MF_F32 ? 4 : 2;
    return (char*)(a.partials + slot * (16 * (int64_t)(a.part_dstride + 2))) +
           ((int64_t)col * a.part_dstride + elem) * ES;
}
__device__ __forceinline__ float* partial_ml(const AttnArgs& a, int64_t slot) {
    return a.partials + slot * (16 * (int64_t)(a.part_dstride + 2)) + 16 * a.part_dstride;
}

// merge_range accumulates partitions p0, p0+pinc, ... relative to their own
// maximum `mx` (lane (g, j): column j, head_dim range [4g*VCH, 4g*VCH+4*VCH)).
// Partitions go four at a time with every load of a batch issued before any
// is used (a batch past the last partition loads only what exists; the
// condition is wave-uniform), and the running maximum moves batch to batch:
// a merge of n partitions per wave costs ceil(n/4) memory round trips. PT: the
// type of the partial outputs; B: partitions per batch.
template <int DT, int DP, int PT = DT, int B = 4>
__device__ __forceinline__ void merge_range(const AttnArgs& a, const int32_t* mg, int p0, int pinc, int j,
                                            int dbase, float& mx, float& L, float (&o)[DP / 4]) {
    constexpr int VCH = DP / 16;
    constexpr int ES = PT == MF_F32 ? 4 : 2;
    constexpr int NW = 4 * VCH * ES / 4;  // words of the lane's chunk
    const int np = mg[3], slot0 = mg[4], sstride = mg[5];
    mx = kMinM;
    L = 0.f;
#pragma unroll
    for (int e = 0; e < 4 * VCH; ++e) o[e] = 0.f;
    for (int p = p0; p < np; p += B * pinc) {
        uint32_t raw[B][NW];
        float mb[B], lb[B];
#pragma unroll
        for (int b = 0; b < B; ++b) {
            if (p + b * pinc < np) {
                const int64_t slot = slot0 + (int64_t)(p + b * pinc) * sstride;
                ld_words<4 * VCH * ES>(partial_out<PT>(a, slot, j, dbase), raw[b]);
                const float* ml = partial_ml(a, slot);
                mb[b] = ml[j];
                lb[b] = ml[16 + j];
            } else {
#pragma unroll
                for (int e = 0; e < NW; ++e) raw[b][e] = 0u;
                mb[b] = kMinM;
                lb[b] = 0.f;
            }
        }
        float bm = mx;
#pragma unroll
        for (int b = 0; b < B; ++b) bm = fmaxf(bm, mb[b]);
        const float keep = __builtin_amdgcn_exp2f(mx - bm);
        L *= keep;
#pragma unroll
        for (int e = 0; e < 4 * VCH; ++e) o[e] *= keep;
#pragma unroll
        for (int b = 0; b < B; ++b) {
            const float wl = __builtin_amdgcn_exp2f(mb[b] - bm) * lb[b];
            L += wl;
#pragma unroll
            for (int e = 0; e < 4 * VCH; ++e) {
                float v;
                if constexpr (PT == MF_F32) v = __uint_as_float(raw[b][e]);
                else v = bits_to_f32<PT>((raw[b][e >> 1] >> (16 * (e & 1))) & 0xffffu);
                o[e] += wl * v;
            }
        }
        mx = bm;
    }
}

// Output row/head of column tile ct's column j, or false for a padding column.
// mg: a merge record (s, h, column tile, parts, slot0, slot stride, first row,
// rows and flag)
__device__ __forceinline__ bool merge_column(const AttnArgs& a, const int32_t* mg, int j, int& prow, int& qhead) {
    const int h = mg[1], ct = mg[2];
    const int row0 = mg[6];
    const int ncols = (mg[7] & ~MF_PLAN_FP32_PARTIALS) * a.G;
    const int cidx = ct * 16 + j;
    if (cidx >= ncols) return false;
    const int r = cidx / a.G;
    prow = row0 + r;
    if (a.row_map) prow = a.row_map[prow];
    qhead = h * a.G + (cidx - r * a.G);
    return true;
}

// Single-wave merge of one record. FP32B: partitions per batch of a record of
// fp32 partials, 0 where the caller's records have none (prefill items).
template <int DT, int DP, int FP32B = 0>
__device__ __forceinline__ void merge_tile(const AttnArgs& a, const int32_t* mg, int g, int j) {
    constexpr int VCH = DP / 16;
    constexpr int ES = DT == MF_F32 ? 4 : 2;
    int prow, qhead;
    const int dbase = 4 * g * VCH;
    if (!merge_column(a, mg, j, prow, qhead) || dbase >= a.head_dim) return;
    float mx, L, o[4 * VCH];
    bool merged = false;
    if constexpr (has_fp32_partials<DT, DP>() && FP32B > 0) {
        if (mg[7] & MF_PLAN_FP32_PARTIALS) {
            merge_range<DT, DP, MF_F32, FP32B>(a, mg, 0, 1, j, dbase, mx, L, o);
            merged = true;
        }
    }
    if (!merged) merge_range<DT, DP>(a, mg, 0, 1, j, dbase, mx, L, o);
    const float inv = L > 0.f ? 1.f / L : 0.f;
#pragma unroll
    for (int e = 0; e < 4 * VCH; ++e) o[e] *= inv;
    store_out_chunk<DT, VCH>(a.out + ((int64_t)prow * a.o_sr + (int64_t)qhead * a.o_sh + dbase) * ES, o);
}

// Fused split-K merge: the last partition of a group to arrive merges the
// group. Release the partials (agent-scope fence: the L2s of the XCDs are not
// coherent with each other), count the arrival, and on the last arrival
// acquire everyone else's partials and reset the counter for the next call.
// Every wave runs to the end; nothing waits on another wave.
template <int DT, int DP>
__device__ __forceinline__ void arrive_and_merge(const AttnArgs& a, int m0, int nct, int lane) {
    if (a.counters == nullptr) return;
    __threadfence();
    int prev = 0;
    if (lane == 0) prev = atomicAdd(a.counters + m0, 1);
    prev = __shfl(prev, 0, 64);
    const int32_t* mg0 = a.merges + (int64_t)m0 * MF_PLAN_MERGE_INTS;
    if (prev == mg0[3] - 1) {
        __threadfence();
        if (lane == 0) a.counters[m0] = 0;
        for (int o = 0; o < nct; ++o) merge_tile<DT, DP>(a, mg0 + o * MF_PLAN_MERGE_INTS, lane >> 4, lane & 15);
    }
}

// -------------------------------------------------------------- main kernel
// Waves per SIMD the register allocator must leave room for: two where the
// kernel fits in 256 registers without spilling (key rows up to 128 bytes,
// or up to 256 bytes for single-tile items), else one. 16-bit wide kernels are
// held to what the shared loop gains from, four (three at 256-byte rows). There
// the whole kernel, with the wave-by-wave body beside the loop, spills at 168
// registers: 61 to 67 vector and 22 to 24 scalar ones, 236 to 244 bytes of
// scratch (50 to 55 vector ones on other block sizes than 16). Compiled without
// that body the loop spills 1 or 2 (9).
#ifndef MF_WIDE_WAVES
#define MF_WIDE_WAVES(dp) ((dp) == 128 ? 3 : 4)
#endif
template <int DT, int DP, int NT>
constexpr int attn_waves_per_eu() {
    constexpr int row_bytes = DP * (DT == MF_F32 ? 4 : 2);
    if (DT != MF_F32 && NT > 1) return MF_WIDE_WAVES(DP);
    return (row_bytes <= 128 || (row_bytes <= 256 && NT == 1)) ? 2 : 1;
}

// Register buffers of the single-column-tile key pipeline: the tile being
// processed plus the two in flight. Measured on MI355X for 128-byte rows
// (bf16 D 64): four and six buffers were no faster than three, and eight
// slower (they cost waves per SIMD); a 256-byte row's buffer is 32 registers,
// and three fit the two-waves-per-SIMD budget.
// One launch for plans holding both single-tile and wide items (see
// attn_mixed_kernel); 0 launches them one after the other.
#ifndef MF_MIXED_LAUNCH
#define MF_MIXED_LAUNCH 1
#endif

// Tiles of extra work the planner charges to the last wave of a cooperative
// unit that holds a multi-row sequence's last tile. Measured on C3's verify
// layer (graph replays): 0 13.2 us, 2 12.96-12.99, 4 12.93-12.94, 6
// 12.36-12.37, 8 12.34-12.37, 10 13.22-13.24, 12 13.18-13.19, 16 13.0. In an
// instrumented build's timeline those waves started their key loop 1.1 us
// after the unit's other waves and ran the boundary and in-flight tiles after
// it, while the others waited at the combine.
#ifndef MF_TAIL_WAVE_TILES
#define MF_TAIL_WAVE_TILES 6
#endif

#ifndef MF_NARROW_DEPTH
#define MF_NARROW_DEPTH 3
#endif

// LDS of the attention kernels: one dynamically sized arena per workgroup.
// A workgroup uses at most one of its two layouts -- the wide items'
// double-buffered K/V stages (workgroup-shared key loop) or the cooperative
// units' softmax states (narrow items) -- so a launch that runs both kinds of
// workgroup (attn_mixed_kernel) sizes the arena for the larger, not for both.
extern __shared__ __attribute__((aligned(16))) char attn_lds[];

// Workgroup-shared prefill loop (attn_wide_body): keys per LDS stage (two
// stage buffers: the stage being computed and the one arriving).
#ifndef MF_WIDE_KEYS
#define MF_WIDE_KEYS(dp) ((dp) == 128 ? 32 : 64)
#endif
constexpr int wide_keys(int dp) { return MF_WIDE_KEYS(dp); }
template <int DT, int DP>
constexpr int wide_lds_bytes() {
    if constexpr (DT == MF_F32) return 0;  // the workgroup-shared loop is 16-bit only
    else return 2 * 2 * wide_keys(DP) * DP * 2;
}
template <int DP>
constexpr int coop_lds_bytes() {
    return (kWaves * 4 * (DP / 16) * 64 + 2 * kWaves * 16) * 4;
}
template <int DT, int DP, int NT, bool FAST>
constexpr int attn_lds_bytes() {
    if constexpr (NT == 1) return coop_lds_bytes<DP>();
    else return wide_lds_bytes<DT, DP>();
}

// The body of one workgroup of the attention kernel: `block` is its index
// among the workgroups that run items of this column-tile width.
// TAIL: a written-in-flight launch (compiled apart, so the other launches
// keep their register budget).
template <int DT, int DP, int NT, bool FAST, bool TAIL = false>
__device__ __forceinline__ void attn_body(const AttnArgs& a, const int block) {
    constexpr int ES = DT == MF_F32 ? 4 : 2;
    constexpr int EPL = 16 / ES;      // elements per 16-byte chunk
    constexpr int NL = DP * ES / 64;  // 16-byte K/Q chunks per lane
    constexpr int VCH = DP / 16;      // V elements per lane per key (= d tiles)
    constexpr int VB = VCH * ES;      // bytes of one lane's V chunk
    constexpr int VWD = VB / 4;       // 32-bit words of one lane's V chunk
    static_assert(NL >= 1 && VWD >= 1, "head_dim too small for this dtype");
    constexpr float kNegInf = -__builtin_huge_valf();

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int item = block * kWaves + wave;
    // The item carries its sequence's first row, row count and kv length (the
    // planner's copies of cu_seqlens / kv_lens), so nothing waits on loading
    // them before the row positions and block table are fetched.
    const int32_t* it = a.items + (int64_t)item * MF_PLAN_ITEM_INTS;
    int4 iv0, iv1, iv2;
    if constexpr (NT == 1) {
        // Single-tile items load their item before the count check, together
        // with the argument block that the check reads (the item list's
        // address needs no argument load when it is preloaded), instead of
        // one round trip after it. The item is in bounds past the live count:
        // plans fill whole workgroups and counted launches size the list by
        // its capacity. The empty asm keeps the loads ahead of the check.
        // Wide items keep the order below: their setup issues the item with
        // the workgroup's other items' keys in one batch after the check.
        iv0 = *(const int4*)it;
        iv1 = *(const int4*)(it + 4);
        iv2 = *(const int4*)(it + 8);
        asm volatile("" ::"s"(iv0.x), "s"(iv0.y), "s"(iv0.z), "s"(iv0.w), "s"(iv1.x), "s"(iv1.y), "s"(iv1.z),
                     "s"(iv1.w), "s"(iv2.x), "s"(iv2.y), "s"(iv2.z), "s"(iv2.w));
        // ... and so do the argument fields the next batch of loads (block
        // table, row positions, Q) is addressed from, which otherwise come
        // from argument cache lines fetched after the check
        asm volatile("" ::"s"(a.block_tables), "s"(a.bt_stride), "s"(a.positions), "s"(a.pool_lens), "s"(a.q),
                     "s"(a.q_sr), "s"(a.q_sh), "s"(a.G), "s"(a.row_map), "s"(a.q_sign));
    }
    const int num_items = a.dev_count ? *a.dev_count : a.num_items;
    if (item >= num_items) return;
    if constexpr (NT != 1) {
        iv0 = make_int4(it[0], it[1], it[2], it[3]);
        iv1 = make_int4(it[4], it[5], it[6], it[7]);
        iv2 = make_int4(it[8], it[9], it[10], it[11]);
    }
    const int lane = threadIdx.x & 63;
    const int g = lane >> 4;  // 16-lane group: MFMA k-group / output row group
    const int j = lane & 15;  // MFMA column (query column) and A-row (key) index

    const int s = iv0.x, h = iv0.y, c0 = iv0.z, nct = iv0.w;
    const int kt0 = iv1.x, kt1 = iv1.y, pslot = iv1.z;
    const int row0 = iv2.x;
    const int ncols = iv2.y * a.G;
    const int kv_len = iv2.z;
    // Keys below pool_len are in the pool; the rest are in-flight rows of the
    // sequence's own new tokens (a verify pass: pool_lens; a written-in-flight
    // step: everything past the keys before the sequence's rows).
    const bool inflight = TAIL || a.pool_lens != nullptr;
    const int pool_len = TAIL ? kv_len - iv2.y : (a.pool_lens != nullptr ? a.pool_lens[s] : kv_len);
    const int D = a.head_dim;

    // The loads that need nothing but the item go out together -- block-table
    // entries first (loads retire in issue order, and the first K/V tiles
    // wait only on them), then row positions, then Q -- so the setup costs
    // one round trip before the K/V stream starts, not three.
    //
    // ---- block-table entries of the item's tiles, two per lane (tile kt0+l
    // and kt0+64+l; fast path, at most kMaxItemTiles), read back with
    // readlane. On a verify pass
    // that is every tile holding a pool key (the boundary tile included);
    // pool_end is the end of the tiles lying wholly in the pool.
    const int tbl_end = inflight ? max(kt0, min(kt1, (pool_len + 15) >> 4)) : kt1;
    const int pool_end = inflight ? max(kt0, min(kt1, pool_len >> 4)) : kt1;
    int tbl = 0, tbl_hi = 0;
    const int tbl_base = kt0;
    if constexpr (FAST) {
        // Every lane loads (a clamped entry past the item's tiles, entry 0 of
        // the row for an item without tiles; only entries of the item's own
        // tiles are ever read back), so no branch skips a load and nothing
        // consumes the values before the other setup loads are issued: the
        // count of loads in flight is the same on every path and later waits
        // stay exact.
        const int idx = kt0 + lane;
        const int32_t* row = a.block_tables + (int64_t)s * a.bt_stride;
        const bool any = tbl_end > kt0;
        tbl = row[any ? min(idx, tbl_end - 1) : 0];
        if constexpr (kMaxItemTiles > 64) tbl_hi = row[any ? min(idx + 64, tbl_end - 1) : 0];
    }
    // physical block of the item's tile i (wave-uniform i)
    auto tbl_at = [&](int i) -> int {
        const int lo = __builtin_amdgcn_readlane(tbl, i & 63);
        if constexpr (kMaxItemTiles > 64) return i < 64 ? lo : __builtin_amdgcn_readlane(tbl_hi, i & 63);
        return lo;
    };

    // ---- columns owned by this lane (one per tile)
    int prow[NT], qhead[NT], qpos[NT];
    bool qvalid[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        // padding columns read row0's position and query (unconditional
        // loads, results discarded)
        const int cidx = (c0 + nt) * 16 + j;
        const bool valid = nt < nct && cidx < ncols;
        const int r = valid ? cidx / a.G : 0;
        const int gq = valid ? cidx - r * a.G : 0;
        int pr = row0 + r;
        if (a.row_map) pr = a.row_map[pr];
        // the low word of the little-endian int64 position (what the int
        // conversion keeps): a 64-bit load's unused high register would be
        // reused as a temporary, and that write waits for the load
        const int pos = reinterpret_cast<const int32_t*>(a.positions)[2 * (int64_t)pr];
        prow[nt] = pr;
        qhead[nt] = h * a.G + gq;
        qpos[nt] = valid ? pos : -1;
        qvalid[nt] = valid;
    }

    // ---- Q fragments (MFMA B operand of S^T = K Q^T): lane (g, j) holds
    // column j's head_dim chunk (c*4 + g) for c < NL.
    uint4 qf[NT][NL];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
#pragma unroll
        for (int c = 0; c < NL; ++c) {
            const int d0 = (c * 4 + g) * EPL;
            // A padding column holds row0's query (its scores are computed
            // and never stored; every column has its own softmax state).
            uint4 v = make_uint4(0, 0, 0, 0);
            if (FAST || d0 < D)  // the fast path has head_dim == DP: every chunk exists
                v = *(const uint4*)(a.q + ((int64_t)prow[nt] * a.q_sr + (int64_t)qhead[nt] * a.q_sh + d0) * ES);
            qf[nt][c] = make_uint4(v.x ^ a.q_sign, v.y ^ a.q_sign, v.z ^ a.q_sign, v.w ^ a.q_sign);
        }
    }

    // General path: address of key `key`'s row for this kv head, or null.
    auto key_row = [&](const char* pool, const char* inflight, int key) -> const char* {
        if (key >= kv_len) return nullptr;
        if (key < pool_len) {
            const int blk = key / a.block_size;
            const int off = key - blk * a.block_size;
            const int phys = a.block_tables[(int64_t)s * a.bt_stride + blk];
            return pool + ((int64_t)phys * a.p_sb + (int64_t)off * a.p_ss + (int64_t)h * a.p_sh) * ES;
        }
        int nr = row0 + (key - pool_len);
        if (a.row_map) nr = a.row_map[nr];
        return inflight + ((int64_t)nr * a.n_sr + (int64_t)h * a.n_sh) * ES;
    };

    // byte offsets of this lane's K chunk (key j, chunk g) and V chunk (keys
    // 4g.., head_dim j*VCH..) inside one block of one kv head
    const uint32_t k_lane_off = (uint32_t)(((int64_t)j * a.p_ss + g * EPL) * ES);
    const uint32_t v_row_bytes = (uint32_t)(a.p_ss * ES);
    const uint32_t v_lane_off = (uint32_t)(((int64_t)(4 * g) * a.p_ss + j * VCH) * ES);
    // Per-key loads of tile kt (the verify boundary and in-flight tiles, and
    // every tile off the fast path). On the fast path a tile's pool keys all
    // lie in one block, whose entry is already in tbl.
    // has_map: the launch has a row map (a compile-time copy of each case:
    // with the map read behind a runtime test, the five row lookups below
    // each ended in a wait for every load in flight, row map or not -- on a
    // verify pass the boundary tile's wave then started its key loop 2.3 us
    // after the others and held up its cooperative unit)
    auto load_general_m = [&](int kt, uint4 (&kf)[NL], uint32_t (&vf)[4][VWD], auto has_map) {
        int phys = 0;
        if constexpr (FAST) phys = kt < tbl_end ? tbl_at(kt - tbl_base) : 0;
        auto row = [&](const char* pool, const char* inflight, int key) -> const char* {
            if constexpr (FAST) {
                if (key >= kv_len) return nullptr;
                if (key < pool_len)
                    return pool + ((int64_t)phys * a.p_sb + (int64_t)(key & 15) * a.p_ss + (int64_t)h * a.p_sh) * ES;
                int nr = row0 + (key - pool_len);
                if constexpr (decltype(has_map)::value) nr = a.row_map[nr];
                return inflight + ((int64_t)nr * a.n_sr + (int64_t)h * a.n_sh) * ES;
            } else {
                return key_row(pool, inflight, key);
            }
        };
        const char* kp = row(a.k_pool, a.new_k, kt * 16 + j);
#pragma unroll
        for (int c = 0; c < NL; ++c) {
            const int d0 = (c * 4 + g) * EPL;
            kf[c] = (kp && d0 < D) ? *(const uint4*)(kp + (int64_t)d0 * ES) : make_uint4(0, 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const char* vp = row(a.v_pool, a.new_v, kt * 16 + 4 * g + r);
            if (vp && j * VCH < D) {
                ld_words<VB>(vp + (int64_t)j * VCH * ES, vf[r]);
            } else {
#pragma unroll
                for (int w = 0; w < VWD; ++w) vf[r][w] = 0;
            }
        }
    };
    auto load_general = [&](int kt, uint4 (&kf)[NL], uint32_t (&vf)[4][VWD]) {
        if (FAST && a.row_map) load_general_m(kt, kf, vf, std::true_type{});
        else load_general_m(kt, kf, vf, std::false_type{});
    };
    // Lane byte offsets of the V rows 4g..4g+3 inside a block, computed once.
    uint32_t v_off[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) v_off[r] = v_lane_off + (uint32_t)r * v_row_bytes;
    // A dummy load (a prefetch slot past the item's last tile) keeps the
    // chunk offsets but drops the lane offsets: the wave reads the block's
    // first few lines instead of the whole tile again. `none` (wave-uniform):
    // the item has no pool tile at all, and the dummy reads the start of Q,
    // which every call has.
    auto load_tile = [&](int kt, uint4 (&kf)[NL], uint32_t (&vf)[4][VWD], bool dummy = false, bool none = false) {
        if constexpr (FAST) {
            // block base is wave-uniform (scalar registers); the lane's byte
            // offsets inside a block never change
            const int phys = tbl_at(kt - tbl_base);
            const int64_t boff = ((int64_t)phys * a.p_sb + (int64_t)h * a.p_sh) * ES;
            const char* kb = none ? a.q : a.k_pool + boff;
            const char* vb = none ? a.q : a.v_pool + boff;
            const uint32_t sel = (dummy || none) ? 0u : 0xffffffffu;
            const uint32_t ko = k_lane_off & sel;
            if constexpr (NT == 1 && DP * ES >= 256) {
                // non-temporal only for rows of 256 bytes or more: measured
                // faster there (bf16 D 128) and slower for 128-byte rows
#pragma unroll
                for (int c = 0; c < NL; ++c) kf[c] = ld_nt16(kb + ko + c * 4 * 16);
#pragma unroll
                for (int r = 0; r < 4; ++r) ld_words_nt<VB>(vb + (v_off[r] & sel), vf[r]);
            } else {
#pragma unroll
                for (int c = 0; c < NL; ++c) kf[c] = *(const uint4*)(kb + ko + c * 4 * 16);
#pragma unroll
                for (int r = 0; r < 4; ++r) ld_words<VB>(vb + (v_off[r] & sel), vf[r]);
            }
        } else {
            load_general(kt, kf, vf);
        }
    };

    // The first NB-1 tiles of a single-column-tile (decode) item go out with
    // the setup loads: positions only trim the item's key range, and these
    // tiles lie in it whenever the item has any. Slots past the item's tiles
    // take a one-line dummy load.
    // The loads are unconditional -- an item without pool tiles issues dummy
    // ones -- so the count of loads in flight is the same on every path and
    // the first use of Q waits for Q alone, not for these tiles too.
    constexpr int NB = NT == 1 ? MF_NARROW_DEPTH : 2;
    uint4 kR[NB][NL];
    uint32_t vR[NB][4][VWD];
    if constexpr (FAST && NT == 1) {
        const bool none = kt0 >= pool_end;
#pragma unroll
        for (int i = 0; i < NB - 1; ++i)
            load_tile(max(kt0, min(kt0 + i, pool_end - 1)), kR[i], vR[i], kt0 + i > pool_end - 1, none);
    }

    int maxpos = -1;
    int minpos = INT_MAX;  // over the item's real columns
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        maxpos = max(maxpos, qpos[nt]);
        if (qvalid[nt]) minpos = min(minpos, qpos[nt]);
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        maxpos = max(maxpos, __shfl_xor(maxpos, off, 64));
        minpos = min(minpos, __shfl_xor(minpos, off, 64));
    }
    minpos = __builtin_amdgcn_readfirstlane(minpos);
    // last key each lane's column may see (-1 for padding columns)
    int lim[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) lim[nt] = qpos[nt] >= 0 ? min(qpos[nt], kv_len - 1) : -1;
    // Tiles past the last key any column may see are never read.
    int kt_end = min(kt1, (min(maxpos, kv_len - 1) >> 4) + 1);
    if (maxpos < 0 || kv_len <= 0) kt_end = kt0;
    kt_end = __builtin_amdgcn_readfirstlane(kt_end);

    // m: running max of the scaled scores (log2 units); thr: the raw score
    // above which a column's running max must move, (m + kLazyLog2) / scale.
    float m[NT], l[NT], thr[NT];
    f32x4 acc[NT][VCH];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        m[nt] = kMinM;
        thr[nt] = (kMinM + kLazyLog2) * a.inv_scale_log2;
        l[nt] = 0.f;
#pragma unroll
        for (int c = 0; c < VCH; ++c) acc[nt][c] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

    // K: lane (g, j) loads key j's head_dim chunks (c*4 + g).
    // V: lane (g, j) loads keys 4g..4g+3, head_dim elements [j*VCH, j*VCH+VCH).
    // FAST path (16-token blocks, head_dim == DP): every
    // load is unconditional, so the compiler can keep the next tile's loads in
    // flight while the current tile is processed.
    // Tiles [kt0, fast_end) run through the pipelined loop. On the fast path
    // with in-flight keys (a verify pass) that is only the tiles lying wholly
    // in the pool; the one or two tiles holding the boundary and the in-flight
    // candidates follow through the general per-key loads.
    int fast_end = kt_end;
    if constexpr (FAST) {
        if (inflight) fast_end = max(kt0, min(kt_end, pool_len >> 4));
    }
    // Per-tile work is branch-free apart from wave-uniform decisions: every
    // column tile's MFMAs run (tiles past nct hold zero queries and are never
    // stored), and masking is a select, so the scheduler sees one straight
    // block per tile, in four parts: scores, the lazy rescale, exponentials
    // and the PV product.
    //
    // Slots past the context in the last block may hold anything, NaN
    // included; p = 0 there, but 0 * NaN is NaN, so clear them.
    auto clear_v_tail = [&](int kt, uint32_t (&vf)[4][VWD]) {
        if constexpr (FAST) {
            if ((kt + 1) * 16 > kv_len) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const bool live = kt * 16 + 4 * g + r < kv_len;
#pragma unroll
                    for (int w = 0; w < VWD; ++w) vf[r][w] = live ? vf[r][w] : 0u;
                }
            }
        }
    };
    // S^T = K Q^T for every column tile (lane (g, j): keys 4g..4g+3 of
    // column j), masked. Scores stay raw; the scale is applied inside the
    // exponent, p = 2^(s * scale - m), one fma.
    auto scores = [&](int kt, const uint4 (&kf)[NL], float (&sv)[NT][4]) {
        f32x4 st[NT];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            st[nt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int c = 0; c < NL; ++c) st[nt] = mfma_qk<DT>(kf[c], qf[nt][c], st[nt]);
        }
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int r = 0; r < 4; ++r) sv[nt][r] = st[nt][r];
        // Every key of a tile wholly inside the context and at or before every
        // column's position is visible to all columns: no mask to apply.
        if (!(kt * 16 + 15 <= minpos && (kt + 1) * 16 <= kv_len)) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    sv[nt][r] = kt * 16 + 4 * g + r <= lim[nt] ? sv[nt][r] : kNegInf;
        }
    };
    // Lazy rescaling: a column's running max m moves (and l, acc are
    // rescaled) only when one of its scores exceeds m by more than
    // kLazyLog2, so p = 2^(s - m) stays below 2^kLazyLog2; l and acc always
    // share the m they were built with, so the result is the same softmax.
    // Each lane tests its own four scores; the max across the column's
    // four lane groups is only formed when some lane asks for a move.
    auto needs_rescale = [&](const float (&sv)[NT][4], float (&lmax)[NT]) -> bool {
        bool grow = false;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            lmax[nt] = fmax_prop(fmax_prop(sv[nt][0], sv[nt][1]), fmax_prop(sv[nt][2], sv[nt][3]));
            grow |= lmax[nt] > thr[nt];
        }
        return __builtin_amdgcn_ballot_w64(grow) != 0;
    };
    auto rescale = [&](const float (&lmax)[NT]) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const float mn = fmaxf(m[nt], group_max4(lmax[nt]) * a.scale_log2);
            const float alpha = __builtin_amdgcn_exp2f(m[nt] - mn);
            l[nt] *= alpha;
#pragma unroll
            for (int c = 0; c < VCH; ++c) acc[nt][c] *= alpha;
            m[nt] = mn;
            thr[nt] = (mn + kLazyLog2) * a.inv_scale_log2;
        }
    };
    // p = 2^(s * scale - m) against the current running max, l += row sums;
    // packed to the 16-bit dtype for the PV MFMA (fp32 kept as is).
    auto exps = [&](const float (&sv)[NT][4], uint2 (&p16)[NT], float (&p32)[NT][4]) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            float p[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) p[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(sv[nt][r], a.scale_log2, -m[nt]));
            l[nt] += (p[0] + p[1]) + (p[2] + p[3]);
            if constexpr (DT == MF_F32) {
#pragma unroll
                for (int r = 0; r < 4; ++r) p32[nt][r] = p[r];
            } else if constexpr (DT == MF_BF16) {
                // hardware round-to-nearest-even pack (v_cvt_pk_bf16_f32)
                p16[nt] = make_uint2(
                    __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){p[0], p[1]}, bf16x2)),
                    __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){p[2], p[3]}, bf16x2)));
            } else {
                p16[nt] = make_uint2(f32_to_bits<DT>(p[0]) | (f32_to_bits<DT>(p[1]) << 16),
                                     f32_to_bits<DT>(p[2]) | (f32_to_bits<DT>(p[3]) << 16));
            }
        }
    };
    // MFMA A operand (16-bit) of head_dim tile c: element c of keys
    // 4g..4g+3, the low (c even) or high halves of word c/2, paired by byte
    // permutes. Row i of tile c is head_dim element i*VCH + c.
    auto va16 = [&](const uint32_t (&vf)[4][VWD], int c) -> uint2 {
        const int wd = c >> 1;
        const uint32_t sel = (c & 1) ? 0x07060302u : 0x05040100u;
        return make_uint2(__builtin_amdgcn_perm(vf[1][wd], vf[0][wd], sel),
                          __builtin_amdgcn_perm(vf[3][wd], vf[2][wd], sel));
    };
    // O^T += V^T P^T for one tile, one MFMA per 16-row head_dim tile c.
    auto pv = [&](const uint32_t (&vf)[4][VWD], const uint2 (&p16)[NT], const float (&p32)[NT][4]) {
#pragma unroll
        for (int c = 0; c < VCH; ++c) {
            if constexpr (DT == MF_F32) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float va = __uint_as_float(vf[r][c]);
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt)
                        acc[nt][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(va, p32[nt][r], acc[nt][c], 0, 0, 0);
                }
            } else {
                const uint2 va = va16(vf, c);
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) acc[nt][c] = mfma_pv16<DT>(va, p16[nt], acc[nt][c]);
            }
        }
    };
    auto process = [&](int kt, const uint4 (&kf)[NL], uint32_t (&vf)[4][VWD]) {
        clear_v_tail(kt, vf);
        float sv[NT][4];
        scores(kt, kf, sv);
        float lmax[NT];
        if (needs_rescale(sv, lmax)) rescale(lmax);
        uint2 p16[NT];
        float p32[NT][4];
        exps(sv, p16, p32);
        pv(vf, p16, p32);
    };

    // ---- key loops. Single-column-tile items (decode, verify) stream their
    // own tiles through the NB-buffer register ring below; wide items pooled
    // four to a workgroup with unrelated items stream theirs through two
    // buffers (attn_wide_body runs the ones that share a key range). Every
    // prefetch is unconditional (past the end it is a dummy or a clamped
    // re-read) because a conditional load makes the compiler drain every
    // outstanding load at the join and serialises the pipeline.
    // The first tile past the pipelined range (a verify pass's boundary or
    // candidate tile) is fetched before the loop, so its per-key loads
    // overlap the pool tiles instead of following them.
    uint4 kT[NL];
    uint32_t vT[4][VWD];
    if constexpr (FAST && NT == 1) {
        if (fast_end < kt_end) load_general(fast_end, kT, vT);
    }
    if (kt0 < fast_end) {
        // Ring of NB register buffers: each step issues the tile NB-1 ahead
        // into the slot freed last and processes the oldest. The loop runs
        // whole rounds of NB steps and the last n % NB tiles (already in
        // slots 0..) follow after it: an exit from inside a round would give
        // the loop a latch that some paths reach with a slot's loads still
        // in flight, and the compiler then drains every load at the top of
        // each round. Prefetches past the last tile still issue (a
        // conditional load would drain the pipeline as well), but as a
        // single line: for 256-byte rows these loads bypass L2, so a full
        // re-read would cost HBM.
        const int last = fast_end - 1;
        int kt = kt0;
        if constexpr (NT == 1) {
            if constexpr (!FAST) {
                // (fast items issued these with the setup loads)
#pragma unroll
                for (int i = 0; i < NB - 1; ++i) load_tile(min(kt0 + i, last), kR[i], vR[i]);
            }
            for (int r = (fast_end - kt0) / NB; r > 0; --r) {
#pragma unroll
                for (int u = 0; u < NB; ++u) {
                    const int nx = kt + NB - 1;
                    load_tile(min(nx, last), kR[(u + NB - 1) % NB], vR[(u + NB - 1) % NB], nx > last);
                    process(kt, kR[u], vR[u]);
                    ++kt;
                }
            }
            // The last (n mod NB) tiles, as nested tests: the flat form (one
            // test per slot) keeps every slot live through the tail and
            // spills at 256-byte rows.
            auto tail = [&](auto self, auto U) {
                constexpr int u = decltype(U)::value;
                if constexpr (u < NB - 1) {
                    if (kt + u <= last) {
                        process(kt + u, kR[u], vR[u]);
                        self(self, std::integral_constant<int, u + 1>{});
                    }
                }
            };
            tail(tail, std::integral_constant<int, 0>{});
        } else {
            // wide items without LDS sharing (a few pooled workgroups): two
            // buffers, which keeps the D 64 kernel at four waves per SIMD
            load_tile(kt, kR[0], vR[0]);
            for (;;) {
                load_tile(min(kt + 1, last), kR[1], vR[1]);
                process(kt, kR[0], vR[0]);
                if (++kt > last) break;
                load_tile(min(kt + 1, last), kR[0], vR[0]);
                process(kt, kR[1], vR[1]);
                if (++kt > last) break;
            }
        }
    }

    if constexpr (FAST) {
        int kt = fast_end;
        if constexpr (NT == 1) {
            if (kt < kt_end) process(kt++, kT, vT);
        }
        for (; kt < kt_end; ++kt) {
            load_general(kt, kR[0], vR[0]);
            process(kt, kR[0], vR[0]);
        }
    }

    // ---- cooperative items: the workgroup's four waves took consecutive key
    // ranges of one (sequence, kv head, column tile) and combine their
    // softmax states through LDS. Every lane (g, j) of every wave holds the
    // same column j and head_dim elements (4g + r)*VCH + c; wave w combines
    // the elements with r == w across the four waves and stores them -- the
    // normalised output, or one partial of a longer split.
    if constexpr (NT == 1) {
        if (iv2.w != 0) {  // the planner flags all four items of a cooperative workgroup
            static_assert(coop_lds_bytes<DP>() == (kWaves * 4 * VCH * 64 + 2 * kWaves * 16) * 4, "LDS arena layout");
            auto s_acc = reinterpret_cast<float (*)[4 * VCH][64]>(attn_lds);
            auto s_m = reinterpret_cast<float (*)[16]>(attn_lds + kWaves * 4 * VCH * 64 * 4);
            auto s_l = reinterpret_cast<float (*)[16]>(attn_lds + (kWaves * 4 * VCH * 64 + kWaves * 16) * 4);
            const float lt = group_sum4(l[0]);
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int c = 0; c < VCH; ++c) s_acc[wave][r * VCH + c][lane] = acc[0][c][r];
            if (g == 0) {
                s_m[wave][j] = m[0];
                s_l[wave][j] = lt;
            }
            __syncthreads();
            float mw[kWaves], M = kMinM;
#pragma unroll
            for (int u = 0; u < kWaves; ++u) {
                mw[u] = s_m[u][j];
                M = fmaxf(M, mw[u]);
            }
            float L = 0.f, o[VCH];
#pragma unroll
            for (int c = 0; c < VCH; ++c) o[c] = 0.f;
#pragma unroll
            for (int u = 0; u < kWaves; ++u) {
                const float w = __builtin_amdgcn_exp2f(mw[u] - M);
                L += s_l[u][j] * w;
#pragma unroll
                for (int c = 0; c < VCH; ++c) o[c] += w * s_acc[u][wave * VCH + c][lane];
            }
            const int d0 = (4 * g + wave) * VCH;
            if (nct > 0 && qpos[0] >= 0) {
                if (pslot < 0) {
                    if (d0 < D) {
                        const float inv = L > 0.f ? 1.f / L : 0.f;
#pragma unroll
                        for (int c = 0; c < VCH; ++c) o[c] *= inv;
                        store_elems<DT, VCH>(a.out + ((int64_t)prow[0] * a.o_sr + (int64_t)qhead[0] * a.o_sh + d0) * ES, o);
                    }
                } else {
                    const float inv = L > 0.f ? 1.f / L : 0.f;
#pragma unroll
                    for (int c = 0; c < VCH; ++c) o[c] *= inv;
                    bool fp32 = false;
                    if constexpr (has_fp32_partials<DT, DP>()) fp32 = (iv1.w & MF_PLAN_FP32_PARTIALS) != 0;
                    if (fp32) store_elems<MF_F32, VCH>(partial_out<MF_F32>(a, pslot, j, d0), o);
                    else store_elems<DT, VCH>(partial_out<DT>(a, pslot, j, d0), o);
                    if (g == 0 && wave == 0) {
                        float* ml = partial_ml(a, pslot);
                        ml[j] = M;
                        ml[16 + j] = L;
                    }
                }
            }
            // fused split-K merge: every wave releases its part of the
            // partial, then wave 0 counts the workgroup's arrival
            if (pslot >= 0 && a.counters != nullptr) {
                __threadfence();
                __syncthreads();
                if (wave == 0) {
                    const int m0 = iv1.w & ~MF_PLAN_FP32_PARTIALS;
                    int prev = 0;
                    if (lane == 0) prev = atomicAdd(a.counters + m0, 1);
                    prev = __shfl(prev, 0, 64);
                    const int32_t* mg0 = a.merges + (int64_t)m0 * MF_PLAN_MERGE_INTS;
                    if (prev == mg0[3] - 1) {
                        __threadfence();
                        if (lane == 0) a.counters[m0] = 0;
                        merge_tile<DT, DP, 2>(a, mg0, g, j);
                    }
                }
            }
            return;
        }
    }

    // ---- finish: the lane holds O^T[d = (4g + r)*VCH + c][column j], i.e. the
    // contiguous head_dim range [4g*VCH, 4g*VCH + 4*VCH) of its column.
    const int dbase = 4 * g * VCH;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const float lt = group_sum4(l[nt]);
        if (nt >= nct || qpos[nt] < 0) continue;
        if (pslot < 0) {
            if (dbase < D) {
                const float inv = lt > 0.f ? 1.f / lt : 0.f;
                float vals[4 * VCH];
#pragma unroll
                for (int r = 0; r < 4; ++r)
#pragma unroll
                    for (int c = 0; c < VCH; ++c) vals[r * VCH + c] = acc[nt][c][r] * inv;
                char* op = a.out + ((int64_t)prow[nt] * a.o_sr + (int64_t)qhead[nt] * a.o_sh + dbase) * ES;
                store_out_chunk<DT, VCH>(op, vals);
            }
        } else {
            const float inv = lt > 0.f ? 1.f / lt : 0.f;
            float vals[4 * VCH];
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int c = 0; c < VCH; ++c) vals[r * VCH + c] = acc[nt][c][r] * inv;
            store_out_chunk<DT, VCH>(partial_out<DT>(a, pslot + nt, j, dbase), vals);
            if (g == 0) {
                float* ml = partial_ml(a, pslot + nt);
                ml[j] = m[nt];
                ml[16 + j] = lt;
            }
        }
    }

    if (pslot >= 0) arrive_and_merge<DT, DP>(a, iv1.w, nct, lane);
}

// ------------------------------------------------- workgroup-shared wide items
typedef __attribute__((ext_vector_type(16))) float f32x16;

// S^T / O^T block: 32 rows x 32 columns, contraction over 16 elements (8 per
// lane half).
template <int DT>
__device__ __forceinline__ f32x16 mfma32(uint4 a, uint4 b, f32x16 c) {
    if constexpr (DT == MF_BF16)
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                       0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c,
                                                      0, 0, 0);
}

// 4 keys x 16 head_dim elements per 16-lane group, transposed on the way out
// of LDS: lane i of the group gets element i of the four rows.
__device__ __forceinline__ uint2 ld_tr16(const char* lds) {
    typedef __attribute__((address_space(3))) i16x4 lds_i16x4;
    return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)lds));
}

// ld_lds16 from a wave-uniform base and a 32-bit lane offset: no vector
// address arithmetic per load. The five wait states cover a base that a vector
// instruction (v_readfirstlane) wrote just before, which the compiler cannot
// see to do inside the assembly, and the m0 write's one.
__device__ __forceinline__ void ld_lds16_base(const char* base_, uint32_t lane_off, uint32_t lds_addr) {
    const uint64_t u = (uint64_t)(uintptr_t)base_;
    const uint64_t base = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)u) |
                          ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(u >> 32)) << 32);
    asm volatile("s_nop 4\n\tglobal_load_lds_dwordx4 %1, %2" ::"{m0}"(lds_addr), "v"(lane_off), "s"(base) : "memory");
}

// A workgroup whose four wide items are column groups of one (sequence, kv
// head, key range): each wave owns 32 columns, and every K/V row of the range
// is staged in LDS once for the four waves.
//
// Per 32 keys the wave forms S^T = K Q^T and O^T += V^T P^T as 32x32x16 MFMA
// blocks (the full-rate shape: 1.85 PFLOP/s over the chip on this card against
// 1.17 for 16x16x32 and half that for 16x16x16). S^T leaves lane (half hf,
// column c) with keys 8b + 4hf + r of its column; P^T's B operand takes those
// registers as they are, and V^T's A operand is read in the same key order by
// the transposing LDS read, so neither P nor V moves between lanes.
//
// Stages of 64 keys (32 at 256-byte rows) go from global memory straight into
// LDS (two buffers, one barrier per stage). Each wave loads the same few 1 KB pieces of every
// 16-key block, so a piece is one scalar base plus a lane offset that never
// changes: new rows of a written-in-flight step are just another base and
// offset. K rows are xor-swizzled by key in 16-byte chunks (32 keys x one
// chunk read conflict-free), V rows by key mod 4 in pairs of 32-byte granules
// (the transposing read's four rows x 64 bytes hit distinct banks): the
// conflict counter reads zero.
//
// Measured on MI355X against the 16x16 loop this replaces (one layer, KV write
// and merge included): two chunks of 2048 rows after up to 6144 keys, 40/8
// heads x 128, 333 GFLOP: 817 -> 388 us (860 TFLOP/s); 16 prompts of up to 1024
// tokens, 15/5 heads x 64: 32.9 -> 29.1 us. What bounds it: MFMA is busy a third
// of the time and the VALU (exponentials, maxima, packing) as long, in turn
// rather than together -- timing copies without the exponentials, the PV
// products or the LDS reads each gained 10-25%, none more. So waves per SIMD
// count: at 256-byte rows 32-key stages leave room for three (168 registers,
// with spills, and 32 KB of LDS a workgroup), 373 us against 403 with two and
// 64-key stages;
// two score chains at a time took 430 against 436. Scalar registers count too:
// a base computed for every load apart, with a branch each, took 630 us.
//
// Blocks of another size than 16 tokens (BLK16 false) change only where a stage's
// rows are read from: each lane looks up the block of its own key, one stage
// ahead. The planner cuts wide work for workgroups that share their tiles and
// does not see the block size; run wave by wave, its plans took up to 1.7 times
// as long there as the narrower per-wave ranges of the 16x16 loop. Graph
// replays, us, 32-token blocks, that loop, wave by wave, and this: 12 verifies
// of 8 rows at 15/5 heads x 64 33, 50, 20; 6 prompts of up to 900 at 8/2 x 32
// 24, 39, 13; chunks of 512 and 700 after 2000 and 500 at 40/8 x 128 295, 302, 88.
//
// cols holds the first column tile and the tile count of the workgroup's four
// items, in scalar registers: only the block table's round trip stands before
// the first stage. Two to three more did -- the other items' columns by vector
// loads, and a wait for every load in flight behind each test of the row map --
// which beside decode streams cost a mixed step up to 14%. Graph replays, us,
// before and after (and with the 16x16 loop): 2 chunks of 512 rows and 24
// decodes of up to 4700 keys at 15/5 heads x 64 30.6, 26.5 (26.0); 1 chunk of
// 370 and 29 decodes of up to 1150 15.1, 13.6 (13.5); 4 chunks of 512 and 28
// decodes of up to 4096 29.4, 28.7 (31.5); 60 decodes of up to 500 keys and 4
// chunks of about 100 16.0, 15.1 (14.3); 16 prompts of up to 1024 31.5, 30.0
// (35.8). The wave's own item is read again rather than kept: its registers,
// held over the caller's comparison, made the 256-byte kernel spill scalars in
// its loop (two chunks of 2048 rows 409 us against 397).
template <int DT, int DP, bool TAIL, bool BLK16>
__device__ __forceinline__ void attn_wide_body(const AttnArgs& a, const int block,
                                               const int (&cols)[kWaves][2]) {
    constexpr int RB = DP * 2;       // bytes of one key row
    constexpr int NCH = RB / 16;     // 16-byte chunks per row
    constexpr int KEYS = wide_keys(DP), TS = KEYS / 16;  // keys and 16-key blocks per stage
    constexpr int RPB = 256 / RB;    // rows per 256 bytes (all LDS banks once)
    constexpr int NQ = DP / 16;      // MFMA steps of S^T
    constexpr int ND = DP / 32;      // 32-row blocks of O^T
    constexpr int PK = RB / 64;      // 1 KB pieces of 16 K rows (V: as many)
    constexpr int NLD = TS * 2 * PK / 4;  // pieces per wave and stage
    constexpr int NOFF = DP == 128 ? 2 : 1;  // a wave's distinct pieces of a block
    constexpr int HALF = KEYS * RB;     // K rows of a stage, then its V rows
    constexpr int STG = 2 * HALF;
    static_assert(DT != MF_F32 && RPB >= 1 && wide_lds_bytes<DT, DP>() == 2 * STG, "stage layout");
    constexpr float kNegInf = -__builtin_huge_valf();

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int hf = lane >> 5;
    const char *k_pool = a.k_pool, *v_pool = a.v_pool, *new_k = a.new_k, *new_v = a.new_v;
    const int32_t* it = a.items + ((int64_t)block * kWaves + wave) * MF_PLAN_ITEM_INTS;
    const int s = it[0], h = it[1], c0 = it[2], nct = it[3], kt0 = it[4], kt1 = it[5], pslot = it[6], m0 = it[7];
    const int row0 = it[8], nrows = it[9], kv_len = it[10];
    const bool inflight = TAIL || a.pool_lens != nullptr;
    const int pool_len = TAIL ? kv_len - nrows : (a.pool_lens != nullptr ? a.pool_lens[s] : kv_len);

    // block-table entries of the 64 tiles from tbl_base (one per lane), and of
    // the 64 after them (16-token blocks)
    const int32_t* trow = a.block_tables + (int64_t)s * a.bt_stride;
    const int tbl_end = inflight ? min(kt1, (pool_len + 15) >> 4) : kt1;
    const int tbl_last = max(tbl_end - 1, 0);  // tiles past it are new rows: never read through the table
    int tbl_base = kt0;
    int tbl = 0, tbl_next = 0;
    if constexpr (BLK16) {
        tbl = trow[min(kt0 + lane, tbl_last)];
        tbl_next = trow[min(kt0 + 64 + lane, tbl_last)];
    }
    auto tbl_at = [&](int t) -> int { return __builtin_amdgcn_readlane(tbl, t - tbl_base); };  // wave-uniform t

    // other block sizes: the key this lane fetches with its i-th piece of stage u
    // (clamped to the range and the context, whose last row then stands in: it is
    // masked there), and the entries of the blocks that hold a stage's keys
    const unsigned bsz = (unsigned)a.block_size;
    auto piece_key = [&](int u, int i) -> int {
        const int x = wave + 4 * i;
        const int p = x % (2 * PK);
        const int k16 = (p >= PK ? p - PK : p) * (1024 / RB) + lane * 16 / RB;
        return min(min(kt0 + TS * u + x / (2 * PK), kt1 - 1) * 16 + k16, kv_len - 1);
    };
    auto look = [&](int u, int (&phys)[NLD]) {
        if constexpr (!BLK16) {
#pragma unroll
            for (int i = 0; i < NLD; ++i)
                phys[i] = trow[(unsigned)max(min(piece_key(u, i), pool_len - 1), 0) / bsz];
        }
    };
    int ph0[NLD], ph1[NLD];
    look(0, ph0);
    look(1, ph1);

    // ---- this lane's column: position and query (padding columns read
    // row0's and are never stored)
    const int ct = (lane & 31) >> 4, j = lane & 15;
    const int cidx = c0 * 16 + (lane & 31);
    const bool valid = ct < nct && cidx < nrows * a.G;
    const int col = valid ? cidx : 0;
    const int crow = (int)((unsigned)col / (unsigned)a.G);
    const int qhead = h * a.G + col - crow * a.G;
    // its own row and those of the workgroup's other columns (two per lane),
    // whose positions say how far the stages run, without an exchange between
    // the waves. One test of the row map for all three: each one joins behind a
    // wait for every load in flight.
    int rows[3] = {row0 + crow, row0, row0};
    bool other[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int c = (hf ? cols[2 * k + 1][0] : cols[2 * k][0]) * 16 + (lane & 31);
        other[k] = ct < (hf ? cols[2 * k + 1][1] : cols[2 * k][1]) && c < nrows * a.G;
        rows[1 + k] = row0 + (int)((unsigned)(other[k] ? c : 0) / (unsigned)a.G);
    }
    if (!TAIL && a.row_map) {
#pragma unroll
        for (int k = 0; k < 3; ++k) rows[k] = a.row_map[rows[k]];
    }
    int rpos[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) rpos[k] = reinterpret_cast<const int32_t*>(a.positions)[2 * (int64_t)rows[k]];
    const int prow = rows[0];
    const int qpos = valid ? rpos[0] : -1;
    const int wpos = max(other[0] ? rpos[1] : -1, other[1] ? rpos[2] : -1);
    uint4 qf[NQ];
#pragma unroll
    for (int c = 0; c < NQ; ++c) {
        const uint4 v = *(const uint4*)(a.q + ((int64_t)prow * a.q_sr + (int64_t)qhead * a.q_sh + c * 16 + hf * 8) * 2);
        qf[c] = make_uint4(v.x ^ a.q_sign, v.y ^ a.q_sign, v.z ^ a.q_sign, v.w ^ a.q_sign);
    }

    // ---- stages
    const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)attn_lds;
    uint32_t off[NOFF], ioff[NOFF];  // this lane's 16 bytes inside a 16-key block: pool rows, new rows
#pragma unroll
    for (int n = 0; n < NOFF; ++n) {
        const int p = (wave + 4 * n) % (2 * PK);
        const bool isv = p >= PK;
        const int k16 = (isv ? p - PK : p) * (1024 / RB) + lane * 16 / RB;
        const int swz = isv ? ((k16 & 3) / RPB) << 2 : (k16 / RPB) & (NCH - 1);
        const uint32_t piece = (uint32_t)(((lane & (NCH - 1)) ^ swz) << 4);
        off[n] = (uint32_t)(k16 * a.p_ss * 2) + piece;
        ioff[n] = (uint32_t)(k16 * a.n_sr * 2) + piece;
    }
    const int64_t blk_bytes = a.p_sb * 2;
    const char* kp_h = k_pool + (int64_t)h * a.p_sh * 2;  // this kv head's rows
    const char* nk_h = new_k + ((int64_t)(row0 - pool_len) * a.n_sr + (int64_t)h * a.n_sh) * 2;
    const int64_t v_delta = v_pool - k_pool, nv_delta = new_v - new_k;
    const int64_t tile_bytes = 16 * a.n_sr * 2;
    // tiles the fetches clamp to: the item's range for the first stage, the
    // workgroup's last read tile once the positions are in
    int fetch_end = kt1;
    auto fetch = [&](int u, int buf, const int (&phys)[NLD]) __attribute__((always_inline)) {
        const int t0 = kt0 + TS * u;
        if constexpr (!BLK16) {
#pragma unroll
            for (int i = 0; i < NLD; ++i) {
                const int x = wave + 4 * i;
                const int b = x / (2 * PK), p = x % (2 * PK);
                const bool isv = p >= PK;
                const int k16 = (isv ? p - PK : p) * (1024 / RB) + lane * 16 / RB;
                const int swz = isv ? ((k16 & 3) / RPB) << 2 : (k16 / RPB) & (NCH - 1);
                const int key = piece_key(u, i);
                const char* src;
                if (!inflight || key < pool_len) {
                    src = k_pool + (isv ? v_delta : 0) + ((int64_t)phys[i] * a.p_sb +
                                                          (int64_t)((unsigned)key % bsz) * a.p_ss + (int64_t)h * a.p_sh) * 2;
                } else {
                    int nr = row0 + key - pool_len;
                    if (a.row_map) nr = a.row_map[nr];
                    src = new_k + (isv ? nv_delta : 0) + ((int64_t)nr * a.n_sr + (int64_t)h * a.n_sh) * 2;
                }
                ld_lds16(src + (((lane & (NCH - 1)) ^ swz) << 4),
                         lds_base + (uint32_t)(buf * STG + b * 16 * RB + (isv ? HALF + (p - PK) * 1024 : p * 1024)));
            }
            return;
        }
        if (t0 - tbl_base >= 64) {
            tbl_base += 64;
            tbl = tbl_next;
            tbl_next = trow[min(tbl_base + 64 + lane, tbl_last)];
        }
        const uint32_t dst0 = lds_base + (uint32_t)(buf * STG);
        const int key1 = (t0 + TS) * 16;
        const bool whole = t0 + TS <= fetch_end;
        // A stage wholly in the pool or wholly of new rows takes a scalar base
        // per block; the boundary stage, the range's last one, and rows behind
        // a row map take the general form below.
        const bool in_pool = whole & (!inflight | (key1 <= pool_len));
        const bool in_new = whole & inflight & (t0 * 16 >= pool_len) & (key1 <= kv_len) & (a.row_map == nullptr);
        auto piece = [&](int i, const char* block_base, int64_t to_v, uint32_t lane_off) {
            const int p = (wave + 4 * i) % (2 * PK), b = (wave + 4 * i) / (2 * PK);
            const bool isv = p >= PK;
            ld_lds16_base(block_base + (isv ? to_v : 0), lane_off,
                          dst0 + (uint32_t)(b * 16 * RB + (isv ? HALF + (p - PK) * 1024 : p * 1024)));
        };
        if (in_pool) {
#pragma unroll
            for (int i = 0; i < NLD; ++i)
                piece(i, kp_h + (int64_t)tbl_at(t0 + (wave + 4 * i) / (2 * PK)) * blk_bytes, v_delta, off[i % NOFF]);
        } else if (in_new) {
#pragma unroll
            for (int i = 0; i < NLD; ++i)
                piece(i, nk_h + (t0 + (wave + 4 * i) / (2 * PK)) * tile_bytes, nv_delta, ioff[i % NOFF]);
        } else {
#pragma unroll 1
            for (int i = 0; i < NLD; ++i) {
                const int x = wave + 4 * i;
                const int b = x / (2 * PK), p = x % (2 * PK);
                const bool isv = p >= PK;
                const int t = min(t0 + b, fetch_end - 1);
                const uint32_t dst = dst0 + (uint32_t)(b * 16 * RB + (isv ? HALF + (p - PK) * 1024 : p * 1024));
                const int k16 = (isv ? p - PK : p) * (1024 / RB) + lane * 16 / RB;
                const int swz = isv ? ((k16 & 3) / RPB) << 2 : (k16 / RPB) & (NCH - 1);
                const int piece = ((lane & (NCH - 1)) ^ swz) << 4;
                // In a block of the pool every slot exists; a new row past the
                // context reads the last one. Either is masked, and its V row
                // cleared.
                const int key = inflight ? min(t * 16 + k16, kv_len - 1) : t * 16 + k16;
                const char* src;
                if (!inflight || key < pool_len) {
                    const int64_t blk = tbl_at(t);
                    src = k_pool + (isv ? v_delta : 0) + (blk * a.p_sb + (int64_t)k16 * a.p_ss + (int64_t)h * a.p_sh) * 2;
                } else {
                    int nr = row0 + key - pool_len;
                    if (a.row_map) nr = a.row_map[nr];
                    src = new_k + (isv ? nv_delta : 0) + ((int64_t)nr * a.n_sr + (int64_t)h * a.n_sh) * 2;
                }
                ld_lds16(src + piece, dst);
            }
        }
    };
    if constexpr (MF_WIDE_PRIO > 0) __builtin_amdgcn_s_setprio(MF_WIDE_PRIO);
    if (kt1 > kt0) fetch(0, 0, ph0);

    // ---- the columns' causal limits; tiles past the workgroup's last visible
    // key are not read
    const int end_key = min(kv_len, kt1 * 16);
    const int lim = qpos >= 0 ? min(qpos, end_key - 1) : -1;  // last key the column may see here
    int maxlim = lim, minlim = valid ? lim : INT_MAX, wglim = min(wpos, end_key - 1);
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        maxlim = max(maxlim, __shfl_xor(maxlim, o, 64));
        minlim = min(minlim, __shfl_xor(minlim, o, 64));
        wglim = max(wglim, __shfl_xor(wglim, o, 64));
    }
    maxlim = __builtin_amdgcn_readfirstlane(maxlim);
    minlim = __builtin_amdgcn_readfirstlane(minlim);
    wglim = __builtin_amdgcn_readfirstlane(wglim);
    auto sync = [&]() {
        // this wave's LDS reads and writes are done, then all waves'
        __builtin_amdgcn_s_waitcnt((15) | (3 << 14) | (7 << 4) | (0 << 8));  // lgkmcnt(0)
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    const int wg_end = wglim < kt0 * 16 ? kt0 : (wglim >> 4) + 1;
    fetch_end = wg_end;
    const int nst = (wg_end - kt0 + TS - 1) / TS;

    float m = kMinM, l = 0.f;
    float thr = (kMinM + kLazyLog2) * a.inv_scale_log2;
    f32x16 acc[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[d][i] = 0.f;

    // lane addresses inside a stage: K rows (key lane & 31), V rows (key 4hf +
    // (lane & 15) / 4 of each group of 8)
    uint32_t kaddr[NQ], vaddr[ND];
#pragma unroll
    for (int c = 0; c < NQ; ++c)
        kaddr[c] = (uint32_t)((lane & 31) * RB + (((2 * c + hf) ^ ((j / RPB) & (NCH - 1))) << 4));
#pragma unroll
    for (int d = 0; d < ND; ++d)
        vaddr[d] = (uint32_t)(HALF + (4 * hf + (j >> 2)) * RB +
                              (((4 * d + 2 * ct + ((j & 3) >> 1)) ^ (((j >> 2) / RPB) << 2)) << 4) + 8 * (j & 1));

    auto tile = [&](const char* stg, int key0) __attribute__((always_inline)) {
        f32x16 st;
#pragma unroll
        for (int i = 0; i < 16; ++i) st[i] = 0.f;
#pragma unroll
        for (int c = 0; c < NQ; ++c) st = mfma32<DT>(*(const uint4*)(stg + kaddr[c]), qf[c], st);
        if (key0 + 31 > minlim) {
#pragma unroll
            for (int i = 0; i < 16; ++i)
                st[i] = key0 + 8 * (i >> 2) + 4 * hf + (i & 3) <= lim ? st[i] : kNegInf;
        }
        // lazy rescale, as in attn_body; a column's keys lie in two lanes
        float lmax = st[0];
#pragma unroll
        for (int i = 1; i < 16; ++i) lmax = fmax_prop(lmax, st[i]);
        if (__builtin_amdgcn_ballot_w64(lmax > thr) != 0) {
            auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(lmax), __float_as_uint(lmax), false, false);
            const float cm = fmax_prop(__uint_as_float(r[0]), __uint_as_float(r[1]));
            const float mn = fmaxf(m, cm * a.scale_log2);
            const float alpha = __builtin_amdgcn_exp2f(m - mn);
            l *= alpha;
#pragma unroll
            for (int d = 0; d < ND; ++d)
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[d][i] *= alpha;
            m = mn;
            thr = (mn + kLazyLog2) * a.inv_scale_log2;
        }
        uint32_t pw[8];
        float sum = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(st[2 * i], a.scale_log2, -m));
            const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(st[2 * i + 1], a.scale_log2, -m));
            sum += p0 + p1;
            if constexpr (DT == MF_BF16)
                pw[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){p0, p1}, bf16x2));
            else
                pw[i] = f32_to_bits<DT>(p0) | (f32_to_bits<DT>(p1) << 16);
        }
        l += sum;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const uint4 pf = make_uint4(pw[4 * k], pw[4 * k + 1], pw[4 * k + 2], pw[4 * k + 3]);
#pragma unroll
            for (int d = 0; d < ND; ++d) {
                const uint2 v0 = ld_tr16(stg + vaddr[d] + (16 * k) * RB);
                const uint2 v1 = ld_tr16(stg + vaddr[d] + (16 * k + 8) * RB);
                acc[d] = mfma32<DT>(make_uint4(v0.x, v0.y, v1.x, v1.y), pf, acc[d]);
            }
        }
    };

    if (nst > 0) {
        if (nst > 1) fetch(1, 1, ph1);
        const int live_end = min(kv_len, wg_end * 16);  // rows past it may hold anything, NaN included
        if (nst > 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NLD) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        sync();
        look(2, ph0);
        for (int u = 0; u < nst; ++u) {
            char* stg = attn_lds + (u & 1) * STG;
            const int key0 = (kt0 + TS * u) * 16;
            if (key0 + KEYS > live_end) {
                // the last stage: p is 0 for its rows past the context, and 0 * NaN is NaN
                const int first = live_end - key0;
                for (int x = first * NCH + (int)threadIdx.x; x < KEYS * NCH; x += 256)
                    *(uint4*)(stg + HALF + x * 16) = make_uint4(0, 0, 0, 0);
                sync();
            }
#pragma unroll
            for (int v = 0; v < KEYS / 32; ++v)
                if (key0 + 32 * v <= maxlim) tile(stg + v * 32 * RB, key0 + 32 * v);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            sync();
            if (u + 2 < nst) {
                fetch(u + 2, u & 1, ph0);
                look(u + 3, ph0);
            }
        }
    } else {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the first stage still lands in this workgroup's LDS
    }

    // ---- finish: lane (hf, column) holds head_dim elements 32d + 8b + 4hf ..
    // + 3; the halves trade blocks so that each lane stores 16 bytes
    auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(l), __float_as_uint(l), false, false);
    const float lt = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    const float inv = lt > 0.f ? 1.f / lt : 0.f;
    char* dst = nullptr;
    if (qpos >= 0)
        dst = pslot < 0 ? a.out + ((int64_t)prow * a.o_sr + (int64_t)qhead * a.o_sh) * 2
                        : partial_out<DT>(a, pslot + ct, j, 0);
#pragma unroll
    for (int d = 0; d < ND; ++d)
#pragma unroll
        for (int b = 0; b < 4; b += 2) {
            uint32_t w[2][2];
#pragma unroll
            for (int e = 0; e < 2; ++e)
#pragma unroll
                for (int k = 0; k < 2; ++k)
                    w[e][k] = f32_to_bits<DT>(acc[d][4 * (b + e) + 2 * k] * inv) |
                              (f32_to_bits<DT>(acc[d][4 * (b + e) + 2 * k + 1] * inv) << 16);
            auto x = __builtin_amdgcn_permlane32_swap(w[0][0], w[1][0], false, false);
            auto y = __builtin_amdgcn_permlane32_swap(w[0][1], w[1][1], false, false);
            if (qpos >= 0) *(uint4*)(dst + (32 * d + 8 * (b + hf)) * 2) = make_uint4(x[0], y[0], x[1], y[1]);
        }
    if (pslot >= 0) {
        if (qpos >= 0 && hf == 0) {
            float* ml = partial_ml(a, pslot + ct);
            ml[j] = m;
            ml[16 + j] = lt;
        }
        arrive_and_merge<DT, DP>(a, m0, nct, lane);
    }
}

// One workgroup of a launch's items. 16-bit wide items share their key range
// through LDS: the planner gives every such workgroup one (sequence, kv head,
// key range); one whose items differ runs them wave by wave. The four items'
// fields are loaded together and compared without short-circuit: chained &&
// made the compiler issue one load per comparison, each behind a full wait,
// which beside a decode workgroup's streams took 12.7 us of a prefill
// workgroup's setup (4.0 us alone).
template <int DT, int DP, int NT, bool FAST, bool TAIL = false>
__device__ __forceinline__ void attn_block(const AttnArgs& a, const int block) {
    if constexpr (DT != MF_F32 && NT > 1) {
        const int num_items = a.dev_count ? *a.dev_count : a.num_items;
        const int32_t* i0 = a.items + (int64_t)block * kWaves * MF_PLAN_ITEM_INTS;
        int32_t key[kWaves][4];
        int cols[kWaves][2];
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            const int32_t* iw = i0 + w * MF_PLAN_ITEM_INTS;
            key[w][0] = iw[0];
            key[w][1] = iw[1];
            key[w][2] = iw[4];
            key[w][3] = iw[5];
            cols[w][0] = iw[2];
            cols[w][1] = iw[3];
        }
        bool same = (FAST || a.head_dim == DP) & ((block + 1) * kWaves <= num_items);
#pragma unroll
        for (int w = 1; w < kWaves; ++w)
            same = same & (key[w][0] == key[0][0]) & (key[w][1] == key[0][1]) & (key[w][2] == key[0][2]) &
                   (key[w][3] == key[0][3]);
        if (same) {
            attn_wide_body<DT, DP, TAIL, FAST>(a, block, cols);
            return;
        }
    }
    attn_body<DT, DP, NT, FAST, TAIL>(a, block);
}

// The item list comes as a separate first argument, which the build has the
// hardware preload into scalar registers: a wave's first item load then
// needs no load of the argument block (see attn_body).
template <int DT, int DP, int NT, bool FAST, bool TAIL = false>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(attn_waves_per_eu<DT, DP, NT>())))
void attn_kernel(const int32_t* items, AttnArgs a) {
    a.items = items;
    if constexpr (TAIL) {
        // the copy workgroups first (measured on the C2 step: 53.7 us per
        // layer against 55.7 with them last)
        const int b = blockIdx.x;
        if (b < a.w_blocks) write_new_rows<DT>(a, b);
        else attn_block<DT, DP, NT, FAST, true>(a, b - a.w_blocks);
    } else {
        attn_block<DT, DP, NT, FAST>(a, blockIdx.x);
    }
}

// In a mixed launch the single-tile (decode) waves start their loads after a
// short sleep, about the time the dispatcher takes to hand out the launch's
// workgroups. Per-workgroup timestamps of the C2 launch showed a prefill
// workgroup beside a decode workgroup spend 14.6 us (median) from its start
// to its first staged tile, against 6.1 us on a CU without one: its setup
// loads (block table, Q, the first K/V stages) queued behind the decode
// waves' streams, while the decode workgroups themselves finished at 14 us
// and the prefill ones at 34-41 us. With the decode waves held back by one
// s_sleep(32) (2,048 cycles) the prefill setup loads go out first: C2 engine
// layer 43.0-43.6 us against 44.6-45.1 (graph replays, alternating builds);
// two to four sleeps gave 43.3-44.1, six 44.9-45.1, nine 46.0-46.4.
#ifndef MF_MIXED_NARROW_SLEEPS
#define MF_MIXED_NARROW_SLEEPS 1
#endif
__device__ __forceinline__ void narrow_start_delay() {
#pragma unroll
    for (int i = 0; i < MF_MIXED_NARROW_SLEEPS; ++i) __builtin_amdgcn_s_sleep(32);
}

// Single-tile and wide items of one plan in one launch: the first
// workgroups run the single-tile items (decode rows: chains of dependent
// loads, latency-bound), the last `wide_blocks` the wide ones (prefill rows:
// MFMA and softmax work), which fill the slots the single-tile workgroups
// leave and overlap their load latency. Two back-to-back launches would leave
// the chip half idle for the length of the shorter one. Measured on the C2
// step (bf16, D 64, 382 single-tile and 900 wide workgroups): 67.9 us per
// layer as two launches, 62.7 us with the wide workgroups first, 58.6 us with
// the single-tile ones first. Each workgroup is entirely one kind, so the
// barriers of either body stay workgroup-uniform.
//
// Occupancy: with 16-bit rows of 128 bytes (D 64) the launch asks
// for four waves per SIMD. Its LDS is one arena sized for the larger of the
// two bodies (32.8 KB at D 64, so four workgroups fit a CU), and the compiler
// then keeps it to 128 registers with a few spills; three waves per SIMD, the
// single-tile body's own need (140 registers), left the C2 step's 1,104
// workgroups in more than one round of three per CU. Measured on the C2
// engine layer as graph replays: 55.1-56.3 us at four, 56.0-57.3 at three.
template <int DT, int DP, int NTW>
constexpr int mixed_waves_per_eu() {
    if constexpr (DT != MF_F32 && DP == 64) return 4;
    else return attn_waves_per_eu<DT, DP, NTW>() < attn_waves_per_eu<DT, DP, 1>() ? attn_waves_per_eu<DT, DP, NTW>()
                                                                                 : attn_waves_per_eu<DT, DP, 1>();
}
template <int DT, int DP, int NTW>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(mixed_waves_per_eu<DT, DP, NTW>())))
void attn_mixed_kernel(AttnArgs narrow, AttnArgs wide, int wide_blocks) {
    const int b = blockIdx.x;
    const int narrow_blocks = (int)gridDim.x - wide_blocks;
    if (b < narrow_blocks) {
        narrow_start_delay();
        attn_body<DT, DP, 1, true>(narrow, b);
    } else {
        attn_block<DT, DP, NTW, true>(wide, b - narrow_blocks);
    }
}

// The written-in-flight form: the copy workgroups first, then the narrow and
// wide ones. One argument block (the wide items differ only in their list):
// the larger body needs the scalar registers a second block would take.
template <int DT, int DP, int NTW>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(mixed_waves_per_eu<DT, DP, NTW>())))
void attn_mixed_tail_kernel(AttnArgs a, const int32_t* wide_items, int wide_num_items,
                            const int32_t* wide_dev_count, int wide_blocks) {
    const int b = blockIdx.x - a.w_blocks;
    const int narrow_blocks = (int)gridDim.x - a.w_blocks - wide_blocks;
    if (b < 0) {
        write_new_rows<DT>(a, blockIdx.x);
    } else if (b < narrow_blocks) {
        narrow_start_delay();
        attn_body<DT, DP, 1, true, true>(a, b);
    } else {
        AttnArgs w = a;
        w.items = wide_items;
        w.num_items = wide_num_items;
        w.dev_count = wide_dev_count;
        attn_block<DT, DP, NTW, true, true>(w, b - narrow_blocks);
    }
}

// ------------------------------------------------------------ decode slices
// A large decode launch as one resident round of waves (mf_attention_plan_slices).
// The plan cuts the concatenated (sequence, 16-key tile) order into equal
// slices; one wave per (slice, kv head) streams the slice's tiles for its head
// and the waves of a slice sit next to each other in the grid (four to a
// workgroup), so every block's rows are read for all kv heads at about the
// same time and no workgroup waits for another to leave. Measured on MI355X
// with a load-only kernel over the C5 block tables: the per-range plan
// (cooperative units: one CU reading one head's quarters, several rounds of
// workgroups) streams at 5.9 TB/s, the same tiles in one round with a
// workgroup per four heads of a range at 6.5-6.8 TB/s. The plan counts one
// workgroup per CU (one wave per SIMD, MF_SLICE_WAVES_PER_CU): with two per
// CU the C5 layer took 521 us against 505, fewer streams keeping the HBM
// busier (three per CU at head_dim 64: 303 against 287 us).
//
// A slice is a list of segments, each one sequence's tiles [kt0, kt1) (a
// whole range or a piece of one; pieces leave split-K partials for the merge
// kernel). Each lane holds eight of the slice's block-table entries (tile
// lane + 64k), so the register ring below runs across segment boundaries
// without a drain: every segment is padded to a multiple of the ring depth
// with dummy tiles (entry stored as ~block: a one-line load, every key
// masked), which keeps the ring's slot of a tile fixed at tile % depth. Lane
// i holds segment i's record and query position, and each segment start
// loads the next segment's query.
constexpr int kSliceRecordInts = MF_SLICE_INTS;
constexpr int kSliceMaxTiles = MF_SLICE_MAX_TILES;        // table entries per lane: tiles / 64
constexpr int kSliceTableRegs = kSliceMaxTiles / 64;
constexpr int kSliceMaxSegments = MF_SLICE_MAX_SEGMENTS;  // one record per lane at set-up
static_assert(kSliceMaxTiles % 64 == 0 && kSliceMaxSegments <= 64, "slice limits");

template <int DT, int DP>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(attn_waves_per_eu<DT, DP, 1>())))
void attn_slice_kernel(AttnArgs a, int num_slices, int hkv) {
    constexpr int ES = DT == MF_F32 ? 4 : 2;
    constexpr int EPL = 16 / ES;
    constexpr int NL = DP * ES / 64;
    constexpr int VCH = DP / 16;
    constexpr int VB = VCH * ES;
    constexpr int VWD = VB / 4;
    constexpr int NB = MF_NARROW_DEPTH;
    constexpr float kNegInf = -__builtin_huge_valf();

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int w = blockIdx.x * kWaves + wave;
    if (w >= num_slices * hkv) return;
    const int sl = w / hkv;
    const int h = w - sl * hkv;
    const int lane = threadIdx.x & 63;
    const int g = lane >> 4;
    const int j = lane & 15;

    // ---- set-up: the slice's segment records, one per lane, then its
    // block-table entries (4 per lane) and the first ring tiles
    const int32_t* hdr = a.items + (int64_t)sl * kSliceRecordInts;
    const int seg0 = hdr[0], nseg = hdr[1], ntiles = hdr[2];
    if (nseg <= 0 || ntiles <= 0) return;  // (the planner makes no empty slice)
    const int32_t* segs = a.items + ((int64_t)num_slices + seg0) * kSliceRecordInts;
    // Lane i keeps segment i's record (and its query position) for the whole
    // slice: a segment start reads it with readlane, no memory wait.
    const int32_t* rec = segs + (int64_t)min(lane, nseg - 1) * kSliceRecordInts;
    const int4 r0 = *(const int4*)rec;        // s, kt0, kt1, row
    const int4 r1 = *(const int4*)(rec + 4);  // kv_len, slot0, pieces, piece
    int tbl[kSliceTableRegs];
    {
        const int len = lane < nseg ? r0.z - r0.y : 0;
        const int plen = (len + NB - 1) / NB * NB;
        int pend = plen;  // inclusive scan of the padded lengths
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int v = __shfl_up(pend, off, 64);
            if (lane >= off) pend += v;
        }
        const int pstart = pend - plen;
#pragma unroll
        for (int k = 0; k < kSliceTableRegs; ++k) {
            const int t = min(lane + 64 * k, ntiles - 1);
            int idx = 0;  // last segment starting at or before t
#pragma unroll
            for (int step = 32; step >= 1; step >>= 1) {
                const int c = idx + step;
                const int ps = __shfl(pstart, min(c, 63), 64);
                if (c < nseg && ps <= t) idx = c;
            }
            const int ts = __shfl(r0.x, idx, 64);
            const int tk0 = __shfl(r0.y, idx, 64);
            const int tlen = __shfl(len, idx, 64);
            const int o = t - __shfl(pstart, idx, 64);
            const bool real = o < tlen;
            const int e = a.block_tables[(int64_t)ts * a.bt_stride + tk0 + (real ? o : tlen - 1)];
            tbl[k] = real ? e : ~e;
        }
    }
    auto tbl_at = [&](int i) -> int {  // wave-uniform i
        const int k = i >> 6;
        const int l = i & 63;
        int e = __builtin_amdgcn_readlane(tbl[0], l);
#pragma unroll
        for (int q = 1; q < kSliceTableRegs; ++q) e = k == q ? __builtin_amdgcn_readlane(tbl[q], l) : e;
        return e;
    };

    const uint32_t k_lane_off = (uint32_t)(((int64_t)j * a.p_ss + g * EPL) * ES);
    const uint32_t v_row_bytes = (uint32_t)(a.p_ss * ES);
    const uint32_t v_lane_off = (uint32_t)(((int64_t)(4 * g) * a.p_ss + j * VCH) * ES);
    uint32_t v_off[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) v_off[r] = v_lane_off + (uint32_t)r * v_row_bytes;
    // Tile i of the slice; `past` (wave-uniform): a prefetch slot beyond the
    // slice's last tile. Dummy and past tiles load one line per chunk.
    auto load_tile = [&](int i, uint4 (&kf)[NL], uint32_t (&vf)[4][VWD], bool past) {
        const int e = tbl_at(i);
        const int phys = e < 0 ? ~e : e;
        const int64_t boff = ((int64_t)phys * a.p_sb + (int64_t)h * a.p_sh) * ES;
        const char* kb = a.k_pool + boff;
        const char* vb = a.v_pool + boff;
        const uint32_t sel = (past || e < 0) ? 0u : 0xffffffffu;
        const uint32_t ko = k_lane_off & sel;
        if constexpr (DP * ES >= 256) {
#pragma unroll
            for (int c = 0; c < NL; ++c) kf[c] = ld_nt16(kb + ko + c * 4 * 16);
#pragma unroll
            for (int r = 0; r < 4; ++r) ld_words_nt<VB>(vb + (v_off[r] & sel), vf[r]);
        } else {
#pragma unroll
            for (int c = 0; c < NL; ++c) kf[c] = *(const uint4*)(kb + ko + c * 4 * 16);
#pragma unroll
            for (int r = 0; r < 4; ++r) ld_words<VB>(vb + (v_off[r] & sel), vf[r]);
        }
    };

    // Query position of lane i's segment; then the first segment's query
    // (MFMA B operand: lane (g, j) holds column j's head_dim chunks c*4 + g;
    // padding columns j >= G read column 0's, whose scores are never stored)
    // and the first ring tiles. A segment loads the next one's query when it
    // starts, so no segment start waits on memory.
    const int lpos = reinterpret_cast<const int32_t*>(a.positions)[2 * (int64_t)r0.w];
    const bool colv = j < a.G;  // decode: one row, columns 0..G-1 are its heads
    const int qhead = h * a.G + (colv ? j : 0);
    uint4 qn[NL];
    auto load_q = [&](int row) {
#pragma unroll
        for (int c = 0; c < NL; ++c)
            qn[c] = *(const uint4*)(a.q + ((int64_t)row * a.q_sr + (int64_t)qhead * a.q_sh + (c * 4 + g) * EPL) * ES);
    };
    load_q(__builtin_amdgcn_readlane(r0.w, 0));
    uint4 kR[NB][NL];
    uint32_t vR[NB][4][VWD];
#pragma unroll
    for (int i = 0; i < NB - 1; ++i) load_tile(min(i, ntiles - 1), kR[i], vR[i], i > ntiles - 1);

    // ---- per-segment state (the lambdas below read it by reference)
    uint4 qf[NL];
    float m, l, thr;
    f32x4 acc[VCH];
    int lim = -1, minpos = -1, key_end = 0;

    auto process = [&](int kt, const uint4 (&kf)[NL], uint32_t (&vf)[4][VWD]) {
        if ((kt + 1) * 16 > key_end) {
            // keys past the segment (padding, or slots past the context,
            // which may hold anything): p = 0 there, and 0 * NaN is NaN
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const bool live = kt * 16 + 4 * g + r < key_end;
#pragma unroll
                for (int x = 0; x < VWD; ++x) vf[r][x] = live ? vf[r][x] : 0u;
            }
        }
        f32x4 st = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < NL; ++c) st = mfma_qk<DT>(kf[c], qf[c], st);
        float sv[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) sv[r] = st[r];
        if (!(kt * 16 + 15 <= minpos && (kt + 1) * 16 <= key_end)) {
#pragma unroll
            for (int r = 0; r < 4; ++r) sv[r] = kt * 16 + 4 * g + r <= lim ? sv[r] : kNegInf;
        }
        // lazy rescale, exactly as the per-range kernel does it
        const float lmax = fmax_prop(fmax_prop(sv[0], sv[1]), fmax_prop(sv[2], sv[3]));
        if (__builtin_amdgcn_ballot_w64(lmax > thr) != 0) {
            const float mn = fmaxf(m, group_max4(lmax) * a.scale_log2);
            const float alpha = __builtin_amdgcn_exp2f(m - mn);
            l *= alpha;
#pragma unroll
            for (int c = 0; c < VCH; ++c) acc[c] *= alpha;
            m = mn;
            thr = (mn + kLazyLog2) * a.inv_scale_log2;
        }
        float p[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) p[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(sv[r], a.scale_log2, -m));
        l += (p[0] + p[1]) + (p[2] + p[3]);
        if constexpr (DT == MF_F32) {
#pragma unroll
            for (int c = 0; c < VCH; ++c)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    acc[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(vf[r][c]), p[r], acc[c], 0, 0, 0);
        } else {
            uint2 p16;
            if constexpr (DT == MF_BF16) {
                p16 = make_uint2(__builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){p[0], p[1]}, bf16x2)),
                                 __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){p[2], p[3]}, bf16x2)));
            } else {
                p16 = make_uint2(f32_to_bits<DT>(p[0]) | (f32_to_bits<DT>(p[1]) << 16),
                                 f32_to_bits<DT>(p[2]) | (f32_to_bits<DT>(p[3]) << 16));
            }
#pragma unroll
            for (int c = 0; c < VCH; ++c) {
                const int wd = c >> 1;
                const uint32_t sel = (c & 1) ? 0x07060302u : 0x05040100u;
                const uint2 va = make_uint2(__builtin_amdgcn_perm(vf[1][wd], vf[0][wd], sel),
                                            __builtin_amdgcn_perm(vf[3][wd], vf[2][wd], sel));
                acc[c] = mfma_pv16<DT>(va, p16, acc[c]);
            }
        }
    };

    const int dbase = 4 * g * VCH;
    int t = 0;  // slice index of the next tile to process
    for (int si = 0; si < nseg; ++si) {
        const int kt0 = __builtin_amdgcn_readlane(r0.y, si);
        const int kt1 = __builtin_amdgcn_readlane(r0.z, si);
        const int row = __builtin_amdgcn_readlane(r0.w, si);
        const int kv_len = __builtin_amdgcn_readlane(r1.x, si);
        const int pos = __builtin_amdgcn_readlane(lpos, si);
#pragma unroll
        for (int c = 0; c < NL; ++c)
            qf[c] = make_uint4(qn[c].x ^ a.q_sign, qn[c].y ^ a.q_sign, qn[c].z ^ a.q_sign, qn[c].w ^ a.q_sign);
        // the next segment's query (the last segment re-reads its own, so
        // every segment issues the same loads)
        load_q(__builtin_amdgcn_readlane(r0.w, min(si + 1, nseg - 1)));
        key_end = min(kv_len, kt1 * 16);
        lim = colv && pos >= 0 ? min(pos, key_end - 1) : -1;
        minpos = pos;
        m = kMinM;
        thr = (kMinM + kLazyLog2) * a.inv_scale_log2;
        l = 0.f;
#pragma unroll
        for (int c = 0; c < VCH; ++c) acc[c] = f32x4{0.f, 0.f, 0.f, 0.f};

        const int seg_start = t;
        const int rounds = (kt1 - kt0 + NB - 1) / NB;
        for (int r = rounds; r > 0; --r) {
#pragma unroll
            for (int u = 0; u < NB; ++u) {
                const int nx = t + NB - 1;
                load_tile(min(nx, ntiles - 1), kR[(u + NB - 1) % NB], vR[(u + NB - 1) % NB], nx > ntiles - 1);
                process(kt0 + (t - seg_start), kR[u], vR[u]);
                ++t;
            }
        }

        // ---- finish the segment: the normalised output, or its partial
        const float lt = group_sum4(l);
        if (colv && pos >= 0) {
            const int slot0 = __builtin_amdgcn_readlane(r1.y, si);
            if (slot0 < 0) {
                const float inv = lt > 0.f ? 1.f / lt : 0.f;
                float vals[4 * VCH];
#pragma unroll
                for (int r = 0; r < 4; ++r)
#pragma unroll
                    for (int c = 0; c < VCH; ++c) vals[r * VCH + c] = acc[c][r] * inv;
                store_out_chunk<DT, VCH>(a.out + ((int64_t)row * a.o_sr + (int64_t)qhead * a.o_sh + dbase) * ES, vals);
            } else {
                const int pslot = slot0 + h * __builtin_amdgcn_readlane(r1.z, si) + __builtin_amdgcn_readlane(r1.w, si);
                const float inv = lt > 0.f ? 1.f / lt : 0.f;
                float vals[4 * VCH];
#pragma unroll
                for (int r = 0; r < 4; ++r)
#pragma unroll
                    for (int c = 0; c < VCH; ++c) vals[r * VCH + c] = acc[c][r] * inv;
                store_out_chunk<DT, VCH>(partial_out<DT>(a, pslot, j, dbase), vals);
                if (g == 0) {
                    float* ml = partial_ml(a, pslot);
                    ml[j] = m;
                    ml[16 + j] = lt;
                }
            }
        }
    }
}

// --------------------------------------------------------------- merge kernel
// A merge launch's record mi, loaded before its count check (record
// min(mi, num_merges - 1): in bounds for every workgroup of the grid), so the
// load goes out with the argument block's instead of one round trip after it;
// the record list's address and num_merges are the preloaded first arguments.
// The argument fields the merge addresses its partials, row map and output
// from are loaded in the same batch. The empty asm keeps the loads ahead of
// the check.
__device__ __forceinline__ void load_merge_record(const AttnArgs& a, const int32_t* merges, int mi, int num_merges,
                                                  int32_t (&mg)[MF_PLAN_MERGE_INTS]) {
    const int32_t* rec = merges + (int64_t)min(mi, num_merges - 1) * MF_PLAN_MERGE_INTS;
    const int4 r0 = *(const int4*)rec, r1 = *(const int4*)(rec + 4);
    asm volatile("" ::"s"(r0.x), "s"(r0.y), "s"(r0.z), "s"(r0.w), "s"(r1.x), "s"(r1.y), "s"(r1.z), "s"(r1.w));
    asm volatile("" ::"s"(a.G), "s"(a.out), "s"(a.o_sr), "s"(a.o_sh), "s"(a.row_map), "s"(a.partials),
                 "s"(a.part_dstride), "s"(a.head_dim));
    mg[0] = r0.x; mg[1] = r0.y; mg[2] = r0.z; mg[3] = r0.w;
    mg[4] = r1.x; mg[5] = r1.y; mg[6] = r1.z; mg[7] = r1.w;
}

// One wave per merge record, each record a workgroup of its own: the wave
// loads its record's partitions four at a time (merge_range) and writes the
// output directly, with no LDS combine or barrier. Measured on MI355X against
// the two earlier forms (four waves per record splitting its partitions and
// combining them in LDS below 128 records, four records per workgroup above):
// C3's verify layer (75 records) 11.36-11.38 us against 12.29-12.40, the C2
// layer (1,955 records) 37.9-38.1 against 38.2-38.3, C5 (824) the same.
template <int DT, int DP>
__global__ __launch_bounds__(64) void merge_kernel(const int32_t* merges, int num_merges, AttnArgs a) {
    const int mi = blockIdx.x;
    int32_t mg[MF_PLAN_MERGE_INTS];
    load_merge_record(a, merges, mi, num_merges, mg);
    if (mi >= (a.dev_count ? *a.dev_count : num_merges)) return;
    const int lane = threadIdx.x & 63;
    merge_tile<DT, DP, (DP > 128 ? 2 : 4)>(a, mg, lane >> 4, lane & 15);
}

// The split-K merge launch: one single-wave workgroup per record.
template <int DT, int DP>
int launch_merge(const AttnArgs& a, const int32_t* merges, int64_t n_merges, hipStream_t stream) {
    hipLaunchKernelGGL((merge_kernel<DT, DP>), dim3((unsigned)n_merges), dim3(64), 0, stream, merges, (int)n_merges,
                       a);
    return check_launch();
}

// TAIL: a written-in-flight launch (16-token blocks and unpadded head_dim
// only: `fast`); its copy workgroups ride in the first launch, or in a
// copy-only launch when there are no items.
template <int DT, int DP, bool TAIL = false>
int launch_attention(AttnArgs a, const int32_t* items, int64_t n_narrow, int64_t n_wide,
                     const int32_t* merges, int64_t n_merges, bool fast, const int32_t* dev_counts,
                     hipStream_t stream) {
    // With arrival counters the attention kernel merges its own partitions;
    // a merges-only call (no items) still runs the separate merge kernel.
    const bool fused = a.counters != nullptr && (n_narrow + n_wide) > 0;
    constexpr int NTW = wide_tiles(DT, DP);
    if constexpr (TAIL) {
        if (!fast) return MF_ERR_UNSUPPORTED;
        if (a.w_blocks > 0 && n_narrow + n_wide == 0) {
            AttnArgs aw = a;
            aw.items = items;
            aw.num_items = 0;
            aw.dev_count = nullptr;
            hipLaunchKernelGGL((attn_kernel<DT, DP, 1, true, true>), dim3((unsigned)a.w_blocks), dim3(256),
                               (attn_lds_bytes<DT, DP, 1, true>()), stream, aw.items, aw);
            if (int st = check_launch()) return st;
        }
    } else {
        a.w_blocks = 0;
    }
#if MF_MIXED_LAUNCH
    if constexpr (NTW > 1 && DT != MF_F32) {
        if (fast && n_narrow > 0 && n_wide > 0) {
            AttnArgs an = a, aw = a;
            an.items = items;
            an.num_items = (int)n_narrow;
            an.dev_count = dev_counts ? dev_counts + 0 : nullptr;
            aw.items = items + n_narrow * MF_PLAN_ITEM_INTS;
            aw.num_items = (int)n_wide;
            aw.dev_count = dev_counts ? dev_counts + 1 : nullptr;
            const int64_t wide_blocks = (n_wide + kWaves - 1) / kWaves;
            const dim3 grid((unsigned)(a.w_blocks + wide_blocks + (n_narrow + kWaves - 1) / kWaves));
            constexpr int lds = attn_lds_bytes<DT, DP, 1, true>() > attn_lds_bytes<DT, DP, NTW, true>()
                                    ? attn_lds_bytes<DT, DP, 1, true>() : attn_lds_bytes<DT, DP, NTW, true>();
            if constexpr (TAIL)
                hipLaunchKernelGGL((attn_mixed_tail_kernel<DT, DP, NTW>), grid, dim3(256), lds, stream, an,
                                   aw.items, aw.num_items, aw.dev_count, (int)wide_blocks);
            else
                hipLaunchKernelGGL((attn_mixed_kernel<DT, DP, NTW>), grid, dim3(256), lds, stream, an, aw,
                                   (int)wide_blocks);
            if (int st = check_launch()) return st;
            n_narrow = n_wide = 0;
            a.w_blocks = 0;
        }
    }
#endif
    if (n_narrow > 0) {
        a.items = items;
        a.num_items = (int)n_narrow;
        a.dev_count = dev_counts ? dev_counts + 0 : nullptr;
        const dim3 grid((unsigned)(a.w_blocks + (n_narrow + kWaves - 1) / kWaves));
        if (fast)
            hipLaunchKernelGGL((attn_kernel<DT, DP, 1, true, TAIL>), grid, dim3(256),
                               (attn_lds_bytes<DT, DP, 1, true>()), stream, a.items, a);
        else if constexpr (!TAIL)
            hipLaunchKernelGGL((attn_kernel<DT, DP, 1, false>), grid, dim3(256), (attn_lds_bytes<DT, DP, 1, false>()),
                               stream, a.items, a);
        if (int st = check_launch()) return st;
        a.w_blocks = 0;
    }
    if constexpr (NTW > 1) {
        if (n_wide > 0) {
            a.items = items + n_narrow * MF_PLAN_ITEM_INTS;
            a.num_items = (int)n_wide;
            a.dev_count = dev_counts ? dev_counts + 1 : nullptr;
            const dim3 grid((unsigned)(a.w_blocks + (n_wide + kWaves - 1) / kWaves));
            if (fast)
                hipLaunchKernelGGL((attn_kernel<DT, DP, NTW, true, TAIL>), grid, dim3(256),
                                   (attn_lds_bytes<DT, DP, NTW, true>()), stream, a.items, a);
            else if constexpr (!TAIL)
                hipLaunchKernelGGL((attn_kernel<DT, DP, NTW, false>), grid, dim3(256),
                                   (attn_lds_bytes<DT, DP, NTW, false>()), stream, a.items, a);
            if (int st = check_launch()) return st;
        }
    } else {
        if (n_wide > 0) return MF_ERR_ARG;  // the plan was made for another dtype
    }
    if (n_merges > 0 && !fused) {
        a.dev_count = dev_counts ? dev_counts + 2 : nullptr;
        if (int st = launch_merge<DT, DP>(a, merges, n_merges, stream)) return st;
    }
    return MF_OK;
}

// A slice plan (mf_attention_plan_slices): one wave per (slice, kv head),
// then the merge of the sequences split across slices.
template <int DT, int DP>
int launch_slices(AttnArgs a, const int32_t* slices, int64_t n_slices, int hkv, const int32_t* merges,
                  int64_t n_merges, hipStream_t stream) {
    if (n_slices > 0) {
        a.items = slices;
        const int64_t waves = n_slices * hkv;
        const dim3 grid((unsigned)((waves + kWaves - 1) / kWaves));
        hipLaunchKernelGGL((attn_slice_kernel<DT, DP>), grid, dim3(256), 0, stream, a, (int)n_slices, hkv);
        if (int st = check_launch()) return st;
    }
    if (n_merges > 0) {
        if (int st = launch_merge<DT, DP>(a, merges, n_merges, stream)) return st;
    }
    return MF_OK;
}

// Padded head_dim the kernels are built for, or 0 if unsupported.
int padded_head_dim(int dtype, int d) {
    if (d <= 0 || (d & (d - 1)) != 0) return 0;  // powers of two only
    if (dtype == MF_F32) {
        if (d > 128) return 0;
        return d < 16 ? 16 : d;
    }
    if (d > 256) return 0;
    return d < 32 ? 32 : d;
}

inline int part_dstride_for(int head_dim) { return head_dim < 32 ? 32 : head_dim; }

}  // namespace
}  // namespace mf

namespace {
// The planner of mf_attention_plan (num_cus 0), mf_attention_plan_device and
// mf_attention_plan_merge_free (cut false).
int attention_plan(int num_seqs, const int32_t* cu_seqlens, const int32_t* kv_lens, int num_q_heads,
                   int num_kv_heads, int head_dim, int dtype, int partition_tiles, int num_cus, bool cut, int32_t* items,
                   int64_t items_capacity, int32_t* merges, int64_t merges_capacity, int64_t* counts) {
    if (num_seqs < 0 || num_q_heads <= 0 || num_kv_heads <= 0 || head_dim <= 0 || !counts)
        return MF_ERR_ARG;
    if (num_q_heads % num_kv_heads) return MF_ERR_ARG;
    if (num_seqs > 0 && (!cu_seqlens || !kv_lens)) return MF_ERR_ARG;
    const int DP = mf::padded_head_dim(dtype, head_dim);
    if (!mf::dtype_ok(dtype) || !DP) return MF_ERR_UNSUPPORTED;
    const int WT = mf::wide_tiles(dtype, DP);
    const int G = num_q_heads / num_kv_heads;
    const int Hkv = num_kv_heads;

    auto col_tiles = [&](int s) -> int {
        const int qlen = cu_seqlens[s + 1] - cu_seqlens[s];
        if (qlen <= 0 || kv_lens[s] <= 0) return 0;
        return (qlen * G + 15) / 16;
    };

    // Key partition sizes, per item class. Single-column-tile (narrow)
    // items get their parallelism from splitting keys: about MF_NARROW_ITEMS
    // items (two to four waves per SIMD), few enough that partials stay
    // small. (Measured on C5: 128-tile partitions, 4,192 items, beat 64-tile
    // ones, 7,320 items: 539 vs 548 us and a merge of 13.5 vs 20 us.) Wide items already
    // come as many column groups, and each split of one costs a 16-column fp32
    // partial per tile written and merged again, so they are split only as far
    // as it takes to reach kWideItems items.
    // Narrow partition: the candidate (a power of two from 4 to
    // kMaxItemTiles tiles per wave) with the least estimated time, where a
    // launch takes the longer of its bandwidth time and its longest wave's
    // chain of tiles, plus the merge launch if any range is split. A range of
    // T > q tiles runs as ceil(T / 4q) units of four waves. Ties go to the
    // longer partition. The constants are fitted to partition sweeps on
    // MI355X (bf16, D 64) timed as HIP-graph replays, i.e. without host
    // submission time: a lone wave's chain costs about 0.53 us per 16-key
    // tile, decode items stream near 5 TB/s, and a split costs about 9 us of
    // merge. Picks: merge-free 32-tile waves for a 64-sequence decode step of
    // 96-1152 keys (17.0 us against 18.5 at 4 tiles), 8 for C3's verify (16.8
    // against 18.5 merge-free at 32), 16 for C2's decodes, 128 on C5.
    auto narrow_partition = [&](int fallback) {
        constexpr double kChainUs = 0.53, kMergeUs = 9.0, kBytesPerUs = 5.0e6;
        const double tile_us = 16.0 * DP * mf::dtype_size(dtype) * 2 / kBytesPerUs;
        int64_t tiles_all = 0;
        for (int s = 0; s < num_seqs; ++s) {
            const int nct = col_tiles(s);
            if (nct && (nct == 1 || WT == 1)) tiles_all += (int64_t)Hkv * nct * ((kv_lens[s] + 15) / 16);
        }
        if (!tiles_all) return fallback;
        int best_q = fallback;
        double best = 1e300;
        for (int q = 4; q <= mf::kMaxItemTiles; q *= 2) {
            int longest = 0;
            bool split = false;
            for (int s = 0; s < num_seqs; ++s) {
                const int nct = col_tiles(s);
                if (!nct || !(nct == 1 || WT == 1)) continue;
                const int T = (kv_lens[s] + 15) / 16;
                if (T <= q) {
                    longest = std::max(longest, T);
                    continue;
                }
                const int units = (T + 4 * q - 1) / (4 * q);
                const int unit = (T + units - 1) / units;
                longest = std::max(longest, (unit + 3) / 4);
                split = split || units > 1;
            }
            const double est = std::max(tiles_all * tile_us, longest * kChainUs) + (split ? kMergeUs : 0.0);
            if (est <= best) {
                best = est;
                best_q = q;
            }
        }
        return best_q;
    };
    int64_t work = 0, wide_units = 0, narrow_units = 0;
    int wide_max_tiles = 0;
    for (int s = 0; s < num_seqs; ++s) {
        const int nct = col_tiles(s);
        if (!nct) continue;
        const bool narrow = nct == 1 || WT == 1;
        const int groups = narrow ? nct : (nct + WT - 1) / WT;
        const int tiles = (kv_lens[s] + 15) / 16;
        work += (int64_t)Hkv * groups * tiles;
        if (narrow) narrow_units += (int64_t)Hkv * groups;
        if (!narrow) {
            wide_units += (int64_t)Hkv * groups;
            wide_max_tiles = std::max(wide_max_tiles, tiles);
        }
    }
    int P = std::min(partition_tiles, mf::kMaxItemTiles);
    int PW = P;
    bool mixed = false;  // a shared launch of narrow and wide items (quad partitions below)
    if (P <= 0) {
        const int64_t target_items = MF_NARROW_ITEMS;
        int64_t want = (work + target_items - 1) / target_items;
        int PA = 4;
        while (PA < want && PA < mf::kMaxItemTiles) PA *= 2;
        P = narrow_partition(PA);
        // wide: the smallest partition (a power of two, at least PA) whose
        // item count stays within the target
        PW = PA;
        if (wide_units > 0) {
            auto wide_items = [&](int q) {
                int64_t n = 0;
                for (int s = 0; s < num_seqs; ++s) {
                    const int nct = col_tiles(s);
                    if (!nct || nct == 1 || WT == 1) continue;
                    n += (int64_t)Hkv * ((nct + WT - 1) / WT) * (((kv_lens[s] + 15) / 16 + q - 1) / q);
                }
                return n;
            };
            while (PW < mf::kMaxItemTiles && PW < wide_max_tiles && wide_items(PW) > MF_WIDE_ITEMS) PW *= 2;
            // Beside wide items the narrow ones run in the same launch
            // (attn_mixed_kernel), where a narrow chain as long as a wide
            // wave's key range is hidden behind the wide waves; longer
            // narrow partitions then only save items and merges. Measured
            // on the C2 step (PW 32): narrow P 16 (the estimate's pick)
            // 58.1-58.9 us per layer, P 32 56.6-56.8, P 64 60.3-60.5;
            // again with the KV write in the launch and the raised prefill
            // priority: P 16 57.0-57.3, P 32 48.9-49.3, P 64 58.1-58.3.
            // The planner does not see the pool's block size: the shared
            // launch needs 16-key blocks, and with other block sizes the two
            // classes run as separate launches, where the raised partition
            // only lengthens the narrow launch's chains (no effect on
            // results, which do not depend on the partition).
            if (MF_MIXED_LAUNCH && WT > 1 && dtype != MF_F32 && head_dim == DP && narrow_units > 0) {
                P = std::max(P, PW);
                mixed = true;
            }
        }
    }

    // Narrow items (one 16-column tile): a (sequence, kv head, column tile)
    // of at most P key tiles is one single-wave item, packed four to a
    // workgroup with other single items. A longer one is cut into balanced
    // units of at most 4P tiles; a unit is a cooperative workgroup whose four
    // waves take consecutive quarters of its tiles and combine their softmax
    // states through LDS, so only ranges of more than 4P tiles leave split-K
    // partials for the merge kernel.
    //
    // Wide items are launched in workgroups of kWaves (one item per wave).
    // A (sequence, kv head, partition) run of at least kWaves column groups
    // fills whole workgroups of its own -- consecutive column groups, the last
    // one padded with empty items (no column tiles) -- so the workgroup shares
    // each K/V tile through LDS. Shorter runs are pooled and packed kWaves to
    // a workgroup, each wave on its own keys.
    const int U = mf::kWaves;
    // Decode steps planned for a device (one row a sequence, one column tile
    // each) that the general partition leaves with fewer than two workgroups
    // per compute unit. Where its longest chain of tiles sets the time,
    // ranges run as cooperative units from a few tiles on: above 4 / 16 / 32
    // tiles with up to one / two / more (sequence, kv head) pairs per compute
    // unit, and always above P, the most a single wave of the general partition
    // takes (a longer range left to one wave would also lose its tiles past P;
    // us as four-wave units, then as single waves: 64 sequences of 256 keys at
    // 15/5 heads x 64 6.4, 8.5; 40 of 256 at 40/8 x 128 12.8, 17.9; 120 of up to
    // 256 at 9/3 x 64 5.1, 8.1). At 256-byte rows a range is cut where the
    // longest holds more than 80 tiles into units of
    // about total / (1.8 x compute units) tiles, at least 32 and at most 72: two
    // workgroups of a unit per compute unit and one round of them. At 128-byte
    // rows, whose tiles chain three times as fast, a step with ranges of more
    // than 100 tiles keeps the general plan, which cuts those well (59 sequences
    // of up to 2800 keys at 9/3 x 64 19.6 us against 22.7 cut as above).
    // Measured, us, general plan then this one: 64 sequences of up to 1152 keys
    // at 15/5 x 64 17.4, 15.3 (units of 64 tiles and merges 19.2); at 40/8 x 128
    // 4 of 8192 to 24576 84, 66 (units of 128 tiles 76, 256 84); 16 of 500 to
    // 4000 73, 45 (uncut 71); 64 of 200 to 3000 119, 70 (uncut 85).
    //
    // Which plan takes less time is estimated from the longest chain one wave
    // runs (a tile takes 0.33 us at 4 KB of K and V, 0.95 at 8 KB and in
    // proportion above), the bytes at 5.5 TB/s, and a merge launch of 4 us. Where
    // the bytes set the general plan's time and the two come out about the same,
    // the general plan is kept if its workgroups fill the compute units evenly
    // (its tiles are at least 0.7 of those that every unit's longest would make);
    // else its last workgroups run on a part-empty chip. Graph replays over pools
    // larger than the caches, us, general plan then this one whatever the
    // estimate: 1 sequence of 1400 keys at 9/3 x 64 8.7, 11.0; 4 of 1400 at 15/5
    // x 64 8.9, 11.0; 2 of about 2000 at 40/8 x 128 13.6, 16.8; 100 of 1400 there
    // 105, 128 (even), 33 of 5000 202, 128 (264 workgroups on 256 units). Over
    // 772 steps of 1 to 200 sequences at seven shapes the choice takes 0.1% more
    // than the better plan on average, and 8 take over 5% more.
    int single_max = P;
    double unit_tiles = 0;  // tiles per unit of a cut range (0: the general partition)
    const auto decode_units = [](int tiles, double per_unit) {
        const int n = std::max(1, (int)std::lround(tiles / per_unit));
        return std::max(n, (tiles + mf::kWaves * mf::kMaxItemTiles - 1) / (mf::kWaves * mf::kMaxItemTiles));
    };
    if (num_cus > 0 && partition_tiles <= 0 && !mixed) {
        int64_t pairs = 0, tiles_all = 0, singles = 0, units = 0;
        int longest = 0;
        bool decode = true;
        for (int s = 0; s < num_seqs; ++s) {
            const int nct = col_tiles(s);
            if (!nct) continue;
            decode = decode && nct == 1 && cu_seqlens[s + 1] - cu_seqlens[s] == 1;
            const int T = (kv_lens[s] + 15) / 16;
            pairs += Hkv;
            tiles_all += (int64_t)Hkv * T;
            longest = std::max(longest, T);
            if (T > P) units += (int64_t)Hkv * ((T + U * P - 1) / (U * P));
            else singles += Hkv;
        }
        const int row_bytes = DP * mf::dtype_size(dtype);
        const bool long_rows = row_bytes >= 256;
        if (decode && units + singles / U < 2 * (int64_t)num_cus && (long_rows || longest <= 100)) {
            const int single = std::min(P, pairs <= num_cus ? 4 : pairs <= 2 * (int64_t)num_cus ? 16 : 32);
            const double per_unit = cut && long_rows && longest > 80
                                        ? std::min(72.0, std::max(32.0, (double)tiles_all / (1.8 * num_cus)))
                                        : 1e9;
            const double tile_us = row_bytes >= 256 ? 0.95 * row_bytes / 256 : 0.33;
            const double bytes_us = (double)tiles_all * 32 * row_bytes / 5.5e6;
            struct Shape {
                double chain_us, us;  // the longest chain's time, the estimate
                double fill;          // tiles over those of a grid of longest workgroups
                bool split;
            };
            auto shape = [&](int alone, auto units_of) {
                int chain = 0, work = 0;
                int64_t waves = 0;
                bool split = false;
                for (int s = 0; s < num_seqs; ++s) {
                    if (!col_tiles(s)) continue;
                    const int T = (kv_lens[s] + 15) / 16;
                    const int n = T <= alone ? 1 : units_of(T);
                    const int unit = (T + n - 1) / n;
                    chain = std::max(chain, T <= alone ? T : (unit + U - 1) / U);
                    work = std::max(work, T <= alone ? U * T : unit);
                    waves += (int64_t)Hkv * (T <= alone ? 1 : U * n);
                    split = split || n > 1;
                }
                const int64_t grid = ((waves + U - 1) / U + num_cus - 1) / num_cus * num_cus;
                return Shape{chain * tile_us, std::max(bytes_us, chain * tile_us) + (split ? 4.0 : 0.0),
                             (double)tiles_all / ((double)grid * std::max(work, 1)), split};
            };
            Shape general = shape(P, [&](int T) { return (T + U * P - 1) / (U * P); });
            if (!cut && general.split) {
                // the plan a merge-free launch gets without the rule: the smallest
                // partition whose units hold the longest range whole
                int q = 4;
                while (U * q < longest && q < mf::kMaxItemTiles) q *= 2;
                general = shape(q, [&](int T) { return (T + U * q - 1) / (U * q); });
            }
            const Shape units_only = shape(single, [&](int T) { return decode_units(T, per_unit); });
            if (units_only.us < 0.995 * general.us ||
                (units_only.us <= 1.2 * general.us && bytes_us >= 0.9 * general.chain_us && general.fill < 0.7)) {
                single_max = single;
                unit_tiles = per_unit;
            }
        }
    }
    auto round_up = [&](int64_t n) { return (n + U - 1) / U * U; };
    // key partitions of sequence s: count, and the start of partition p
    // (narrow cooperative ranges are balanced; the rest are Q-tile strides).
    // A wide range takes as many partitions as PW-tile strides would give,
    // in strides of equal length: the C2 chunks planned prefill-only
    // 34.9-35.3 us against 36.3-36.6 with PW strides (a short last
    // partition).
    auto partitions = [&](int s, bool narrow, int& Q, bool& coop) {
        const int tiles = (kv_lens[s] + 15) / 16;
        coop = narrow && tiles > single_max;
        Q = narrow ? (coop ? U * P : P) : PW;
        if (narrow && unit_tiles > 0) return coop ? decode_units(tiles, unit_tiles) : 1;
        if (!narrow && tiles > PW) {
            const int np = (tiles + PW - 1) / PW;
            Q = (tiles + np - 1) / np;
        }
        return (tiles + Q - 1) / Q;
    };
    auto part_begin = [&](int tiles, int nparts, int Q, bool coop, int p) {
        return coop ? (int)((int64_t)p * tiles / nparts) : std::min(tiles, p * Q);
    };
    // Quad partitions (mixed plans). A sequence whose wide items fill whole
    // workgroups runs as column quads: the kWaves column groups one
    // workgroup holds, over one key range. In a mixed plan each quad takes
    // its own partitions: the tiles its last column sees, cut into
    // round(visible / W) equal ranges, W chosen so that the launch's wide
    // workgroups carry about two rounds' worth per compute unit (the total
    // visible work over 2 x 256 CUs, at least PW). Every wide workgroup then
    // holds about the same work, and each compute unit about two of them
    // beside the narrow ones, all in one resident round. C2 step, engine
    // layer as graph replays: 44.1-44.2 us against 45.8-46.0 with the ranges'
    // partitions (PW 64 strides); 1.5 workgroups per CU 49.3-49.6, 2.5
    // 47.1-47.4, 3 47.5-48.0, 4 53.3-53.5. Plans of wide items only, made without
    // a device, keep the ranges' partitions (there two per CU took the prefill
    // items of the 16x16 loop from 35.1 to 37.9 us). The XCD queues below take a (sequence, kv head)'s quads
    // as one run: the launch fetches 1.09x its algorithmic reads, against
    // 1.65x with each (quad, kv head) dealt alone (0.3 us faster).
    const int kPlanCUs = num_cus > 0 ? num_cus : 256;  // an MI355X has 256 compute units
    // A plan made for a device cuts every wide sequence by quads -- also one of
    // fewer than four column groups, whose quad has idle waves but whose tiles
    // are shared -- and a shared workgroup's range may be any length (its block
    // table is read 64 tiles at a time). At 128-byte rows and less, a plan of
    // wide items only does so where the general ranges come out shorter than 32
    // tiles (PW), and a workgroup's set-up costs more than its tiles: 15/5 heads
    // x 64, device against general ranges, us: 1024 fresh rows (8 tiles) 18.1
    // against 23.9, 8 prompts of up to 300 (4) 14.2 / 18.9, 256 rows after 6144
    // keys (19) 24.3 / 27.7, but 4 chunks of 512 after up to 2048 (32) 25.6 /
    // 28.6 and 16 prompts of up to 1024 (64) 30 / 32. At 256-byte rows it always
    // does: 2 chunks of 2048 after 6144 keys 370 against 428 (10,240 merges).
    const bool device = num_cus > 0 && partition_tiles <= 0 && WT > 1 && dtype != MF_F32 && head_dim == DP &&
                        (mixed || DP >= 128 || PW < 32);
    auto quads = [&](int s) -> int {  // column quads of s, 0 if s is not a shared wide sequence
        const int nct = col_tiles(s);
        if (!(mixed || device) || !nct || nct == 1 || WT == 1) return 0;
        const int ngroups = (nct + WT - 1) / WT;
        return device || ngroups >= U ? (int)(round_up(ngroups) / U) : 0;
    };
    auto quad_visible = [&](int s, int qd) -> int {
        const int rows = cu_seqlens[s + 1] - cu_seqlens[s];
        const int end_ct = std::min(col_tiles(s), (qd + 1) * U * WT);
        const int last_col = std::min(end_ct * 16, rows * G) - 1;
        const int last_pos = kv_lens[s] - rows + last_col / G;
        return std::max(1, std::min((kv_lens[s] + 15) / 16, last_pos / 16 + 1));
    };
    double quad_w = 1.0;
    const int max_range = device ? INT_MAX : mf::kMaxItemTiles;
    if (mixed || device) {
        int64_t visible = 0, quad_units = 0;
        int longest = 0;
        for (int s = 0; s < num_seqs; ++s)
            for (int qd = 0, nq = quads(s); qd < nq; ++qd) {
                const int v = quad_visible(s, qd);
                visible += (int64_t)Hkv * v;
                quad_units += Hkv;
                longest = std::max(longest, v);
            }
        quad_w = std::max((double)std::max(PW, 1), (double)visible / (2.0 * kPlanCUs));
        if (device && !mixed) {
            // About two workgroups per compute unit, of at least 16 tiles (12 at
            // head_dim 128: 7-row verifies of up to 600 keys at 40/8 18.5 us
            // against 21.8 at 16); where that makes ranges longer than 96 tiles, about four, of at
            // least 96. Measured, us at 8 / 16 / 24 / 32 / 48 / 64 / 128 tiles
            // per range and uncut: one chunk of 256 rows after 6144 keys, 15/5
            // heads x 64 33.6 / 27.3 / 24.3 / 24.0 / 24.7 / 29.2 / 38 / 88 (rule
            // 23), 40/8 x 128 99 / 71 / 62 / 66 / 51 / 58 / 79 / 202 (64); 1024
            // fresh rows, x 64 19.8 / 18.1 / 19.1 / 21.4 / 21.0 uncut (16), x 128
            // 50 / 36 / 36 / 41 / 45 uncut (20); 2 chunks of about 850 rows
            // after 4000 keys x 128 714 / 449 / 374 / 335 / 301 / 291 / 295 / 292
            // (200: 284).
            // Short launches: cut in two, their quads run half the chain and
            // then a merge, which costs more than the other half. Whole quads
            // where the longest sees at most 31 tiles; where the (quad, kv head)
            // pairs fill no more than a third of the compute units, at most 21,
            // and above that, up to 95, ranges of 8 tiles that the idle units
            // run beside each other. Graph replays over pools larger than the
            // caches, us at 8 tiles / the floor above / whole: 8-row verifies of
            // up to 450 keys at 15/5 heads x 64, 3 of them 9.9 / 10.2 / 10.2, 16
            // 11.9 / 14.5 / 12.8, 40 12.9 / 14.8 / 12.5; of up to 1000, 8 of them
            // 12.3 / 14.0 / 20; 16 prompts of up to 500 at 9/3 x 64 18.1 / 17.4 /
            // 15.2; 4 of up to 300 at 40/8 x 128 22.7 / 22.4 / 19.0.
            const bool few = quad_units <= kPlanCUs / 3;
            const double floor = longest < (few ? 22 : 32) ? longest : few && longest < 96 ? 8 : DP >= 128 ? 12 : 16;
            quad_w = std::max(floor, (double)visible / (2.0 * kPlanCUs));
            if (quad_w > 96) quad_w = std::max(96.0, (double)visible / (4.0 * kPlanCUs));
        }
    }
    // Partition counts per (sequence, quad), then at most two wide
    // workgroups per CU: rounding can leave a few more, and with every CU
    // holding two, those few land as a third on some CU, which then finishes
    // last. Partitions are merged, one at a time, in the quad whose ranges
    // grow the least. C2: 530 -> 510 workgroups, engine layer 42.1-42.3 us
    // against 42.7-42.9.
    std::vector<std::vector<int>> qparts(num_seqs);
    if (mixed || device) {
        int64_t total = 0;
        for (int s = 0; s < num_seqs; ++s) {
            const int nq = quads(s);
            qparts[s].resize(nq);
            for (int qd = 0; qd < nq; ++qd) {
                const int v = quad_visible(s, qd);
                const int n = std::max(1, (int)std::lround(v / quad_w));
                qparts[s][qd] = std::max<int>(n, ((int64_t)v + max_range - 1) / max_range);
                total += (int64_t)Hkv * qparts[s][qd];
            }
        }
        while (mixed && total > 2 * kPlanCUs) {
            int bs = -1, bq = -1;
            double best = 1e300;
            for (int s = 0; s < num_seqs; ++s)
                for (int qd = 0; qd < (int)qparts[s].size(); ++qd) {
                    const int n = qparts[s][qd], v = quad_visible(s, qd);
                    if (n <= 1 || (v + n - 2) / (n - 1) > max_range) continue;
                    const double grown = (double)v / (n - 1);
                    if (grown < best) {
                        best = grown;
                        bs = s;
                        bq = qd;
                    }
                }
            if (bs < 0) break;  // every quad is down to one range (or at the item limit)
            --qparts[bs][bq];
            total -= Hkv;
        }
    }
    auto quad_parts = [&](int s, int qd) { return qparts[s][qd]; };

    // First walk: sizes only.
    int64_t n_single = 0, n_coop = 0, n_wide = 0, n_loose = 0, n_merges = 0, n_slots = 0;
    for (int s = 0; s < num_seqs; ++s) {
        const int nct = col_tiles(s);
        if (!nct) continue;
        const bool narrow = nct == 1 || WT == 1;
        int Q;
        bool coop;
        const int nparts = partitions(s, narrow, Q, coop);
        const int width = narrow ? 1 : WT;
        const int ngroups = (nct + width - 1) / width;
        if (narrow) {
            if (coop) n_coop += (int64_t)U * nparts * Hkv * ngroups;
            else n_single += (int64_t)nparts * Hkv * ngroups;
        } else if (const int nq = quads(s)) {
            for (int qd = 0; qd < nq; ++qd) {
                const int n = quad_parts(s, qd);
                const int cols = std::min(nct, (qd + 1) * U * WT) - qd * U * WT;
                n_wide += (int64_t)Hkv * n * U;
                if (n > 1) {
                    n_slots += (int64_t)Hkv * n * cols;
                    n_merges += (int64_t)Hkv * cols;
                }
            }
            continue;
        } else if (ngroups >= U) {
            n_wide += (int64_t)nparts * Hkv * round_up(ngroups);
        } else {
            n_loose += (int64_t)nparts * Hkv * ngroups;
        }
        if (nparts > 1) {
            n_slots += (int64_t)Hkv * nparts * nct;
            n_merges += (int64_t)Hkv * nct;
        }
    }
    const int64_t n_narrow = round_up(n_single) + n_coop;
    n_wide += round_up(n_loose);
    const int64_t pstride = 16 * (int64_t)(mf::part_dstride_for(head_dim) + 2);
    counts[0] = n_narrow;
    counts[1] = n_wide;
    counts[2] = n_merges;
    counts[3] = n_slots * pstride;
    if (n_narrow + n_wide > items_capacity || n_merges > merges_capacity) return MF_ERR_WORKSPACE;
    if ((n_narrow + n_wide) > 0 && !items) return MF_ERR_ARG;
    if (n_merges > 0 && !merges) return MF_ERR_ARG;

    // Second walk: stage the items and write the merges. Column group gi of
    // a sequence owns partial slots from slot0 + gi*Hkv*nparts*width
    // (head-major, then partition, then its w tiles) and merge records from
    // merge0 + gi*Hkv*width.
    typedef std::array<int32_t, MF_PLAN_ITEM_INTS> Item;
    std::vector<Item> singles, coop_items, shared_items, loose_items;
    int64_t wm = 0, slots = 0;
    for (int s = 0; s < num_seqs; ++s) {
        const int nct = col_tiles(s);
        if (!nct) continue;
        const bool narrow = nct == 1 || WT == 1;
        const int tiles = (kv_lens[s] + 15) / 16;
        int Q;
        bool coop;
        const int nparts = partitions(s, narrow, Q, coop);
        const int width = narrow ? 1 : WT;
        const int ngroups = (nct + width - 1) / width;
        if (const int nq = narrow ? 0 : quads(s)) {
            // quad partitions: per (kv head, quad), each column group owns
            // n * w consecutive slots (partition-major) and w merge records;
            // a kv head's workgroups are consecutive (one XCD run)
            for (int h = 0; h < Hkv; ++h) {
                for (int qd = 0; qd < nq; ++qd) {
                    const int n = quad_parts(s, qd);
                    const int v = quad_visible(s, qd);
                    int64_t gslot[mf::kWaves], grec[mf::kWaves];
                    for (int k = 0; k < U; ++k) {
                        const int gi = qd * U + k;
                        gslot[k] = grec[k] = -1;
                        if (gi >= ngroups || n <= 1) continue;
                        const int w = std::min(WT, nct - gi * WT);
                        gslot[k] = slots;
                        slots += (int64_t)n * w;
                        grec[k] = wm;
                        for (int o2 = 0; o2 < w; ++o2, ++wm) {
                            int32_t* o = merges + wm * MF_PLAN_MERGE_INTS;
                            o[0] = s;
                            o[1] = h;
                            o[2] = gi * WT + o2;
                            o[3] = n;
                            o[4] = (int32_t)(gslot[k] + o2);
                            o[5] = w;
                            o[6] = cu_seqlens[s];
                            o[7] = cu_seqlens[s + 1] - cu_seqlens[s];
                        }
                    }
                    for (int p = 0; p < n; ++p) {
                        const int k0 = (int)((int64_t)p * v / n);
                        // v counts the keys of distinct positions that end the
                        // context; rows that share a position (the operator's
                        // non-causal queries) see more, so a device plan's last
                        // range runs to the context's end and the kernel stops
                        // where its rows do
                        const int k1 = device && p + 1 == n ? tiles : (int)((int64_t)(p + 1) * v / n);
                        for (int k = 0; k < U; ++k) {
                            const int gi = qd * U + k;
                            Item o{};
                            o[0] = s;
                            o[1] = h;
                            o[4] = k0;
                            o[5] = k1;
                            o[8] = cu_seqlens[s];
                            o[9] = cu_seqlens[s + 1] - cu_seqlens[s];
                            o[10] = kv_lens[s];
                            if (gi < ngroups) {
                                const int w = std::min(WT, nct - gi * WT);
                                o[2] = gi * WT;
                                o[3] = w;
                                o[6] = n > 1 ? (int32_t)(gslot[k] + (int64_t)p * w) : -1;
                                o[7] = n > 1 ? (int32_t)grec[k] : -1;
                            } else {  // padding: same keys, no columns, no partial slot
                                o[2] = (ngroups - 1) * WT;
                                o[6] = -1;
                                o[7] = -1;
                            }
                            shared_items.push_back(o);
                        }
                    }
                }
            }
            continue;
        }
        const int64_t slot0 = slots, merge0 = wm;
        const int32_t fp32_flag = narrow && unit_tiles > 0 && dtype != MF_F32 ? MF_PLAN_FP32_PARTIALS : 0;
        auto make = [&](int gi, int p, int h, int k0, int k1) {
            const int cg0 = gi * width;
            const int w = std::min(width, nct - cg0);
            Item o;
            o[0] = s;
            o[1] = h;
            o[2] = cg0;
            o[3] = w;
            o[4] = k0;
            o[5] = k1;
            o[6] = nparts > 1 ? (int32_t)(slot0 + (int64_t)gi * Hkv * nparts * width + ((int64_t)h * nparts + p) * w)
                              : -1;
            o[7] = nparts > 1 ? (int32_t)(merge0 + (int64_t)gi * Hkv * width + (int64_t)h * w) | fp32_flag : -1;
            o[8] = cu_seqlens[s];
            o[9] = cu_seqlens[s + 1] - cu_seqlens[s];
            o[10] = kv_lens[s];
            o[11] = 0;
            return o;
        };
        for (int p = 0; p < nparts; ++p) {
            const int k0 = part_begin(tiles, nparts, Q, coop, p);
            const int k1 = part_begin(tiles, nparts, Q, coop, p + 1);
            for (int hi = 0; hi < Hkv; ++hi) {
                // A device's decode units start one kv head on from the last
                // range's: with 8 heads workgroup b's head would otherwise be b
                // mod 8, its XCD's number, and an XCD that reads one head of
                // every row uses one channel in eight of its L2 (67 against 75
                // us, the 4 long sequences at 64-tile units).
                const int h = narrow && unit_tiles > 0 ? (hi + p + s) % Hkv : hi;
                if (narrow) {
                    for (int gi = 0; gi < ngroups; ++gi) {
                        if (!coop) {
                            singles.push_back(make(gi, p, h, k0, k1));
                            continue;
                        }
                        // four waves on consecutive quarters of [k0, k1). In
                        // the unit holding a multi-row sequence's last tile (a
                        // verify pass: the boundary tile and the in-flight
                        // candidates, loaded key by key), the last wave counts
                        // MF_TAIL_WAVE_TILES more tiles than it has, so the
                        // others take them and the unit's waves reach its
                        // LDS combine together -- as far as a wave's
                        // block-table registers go.
                        const int n = k1 - k0;
                        const int rows = cu_seqlens[s + 1] - cu_seqlens[s];
                        const int extra = (k1 == tiles && rows > 1)
                                              ? std::min(MF_TAIL_WAVE_TILES, U * mf::kMaxItemTiles - n) : 0;
                        auto cut = [&](int w) {
                            return w >= U ? k1 : std::min(k1, k0 + (int)((int64_t)w * (n + extra) / U));
                        };
                        for (int w = 0; w < U; ++w) {
                            Item o = make(gi, p, h, cut(w), cut(w + 1));
                            o[11] = 1;
                            coop_items.push_back(o);
                        }
                    }
                } else if (ngroups >= U) {
                    for (int gi = 0; gi < round_up(ngroups); ++gi) {
                        Item o = make(std::min(gi, ngroups - 1), p, h, k0, k1);
                        if (gi >= ngroups) {  // padding: same keys, no columns, no partial slot
                            o[3] = 0;
                            o[6] = -1;
                            o[7] = -1;
                        }
                        shared_items.push_back(o);
                    }
                } else {
                    for (int gi = 0; gi < ngroups; ++gi) loose_items.push_back(make(gi, p, h, k0, k1));
                }
            }
        }
        if (nparts > 1) {
            for (int gi = 0; gi < ngroups; ++gi) {
                const int cg0 = gi * width;
                const int w = std::min(width, nct - cg0);
                const int64_t group_base = slot0 + (int64_t)gi * Hkv * nparts * width;
                for (int h = 0; h < Hkv; ++h) {
                    for (int o2 = 0; o2 < w; ++o2) {
                        int32_t* o = merges + wm * MF_PLAN_MERGE_INTS;
                        o[0] = s;
                        o[1] = h;
                        o[2] = cg0 + o2;
                        o[3] = nparts;
                        o[4] = (int32_t)(group_base + (int64_t)h * nparts * w + o2);
                        o[5] = w;
                        o[6] = cu_seqlens[s];
                        o[7] = (cu_seqlens[s + 1] - cu_seqlens[s]) | fp32_flag;
                        ++wm;
                    }
                }
            }
            slots += (int64_t)Hkv * nparts * nct;
        }
    }
    // Longest first: the hardware hands out workgroups in order as slots free
    // up, so the last round of the grid is made of the short remainder
    // partitions instead of a few long ones. Items that run alone are sorted
    // and then cut into workgroups (the last padded with empty items); all
    // workgroups are ordered by their longest item. Stable, so equal lengths
    // keep their heads-adjacent order.
    auto len = [](const Item& o) { return o[5] - o[4]; };
    auto longer = [&](const Item& x, const Item& y) { return len(x) > len(y); };
    auto pad_to_workgroups = [&](std::vector<Item>& v) {
        std::stable_sort(v.begin(), v.end(), longer);
        while (v.size() % U) {
            Item o{};
            o[6] = -1;
            o[7] = -1;
            v.push_back(o);
        }
    };
    auto unit_len = [&](const Item* u) {
        int l = 0;
        for (int w = 0; w < U; ++w) l = std::max(l, len(u[w]));
        return l;
    };
    auto emit = [&](std::vector<const Item*>& units, int64_t wi) {
        std::stable_sort(units.begin(), units.end(),
                         [&](const Item* x, const Item* y) { return unit_len(x) > unit_len(y); });
        for (const Item* u : units)
            for (int w = 0; w < U; ++w, ++wi) std::copy(u[w].begin(), u[w].end(), items + wi * MF_PLAN_ITEM_INTS);
    };
    pad_to_workgroups(singles);
    pad_to_workgroups(loose_items);
    std::vector<const Item*> nunits, wunits;
    for (size_t i = 0; i < coop_items.size(); i += U) nunits.push_back(&coop_items[i]);
    for (size_t i = 0; i < singles.size(); i += U) nunits.push_back(&singles[i]);
    for (size_t i = 0; i < shared_items.size(); i += U) wunits.push_back(&shared_items[i]);
    for (size_t i = 0; i < loose_items.size(); i += U) wunits.push_back(&loose_items[i]);
    emit(nunits, 0);
    // A wide item's work: its tiles up to the last one its last column sees
    // (causal), a workgroup's the most of its four.
    auto item_work = [&](const Item& o) -> int64_t {
        const int ncols = o[9] * G;
        const int last_col = std::min((o[2] + o[3]) * 16, ncols) - 1;
        if (o[3] <= 0 || last_col < 0) return 0;
        const int last_pos = o[10] - o[9] + last_col / G;
        return std::max(0, std::min(o[5], last_pos / 16 + 1) - o[4]);
    };
    auto unit_work = [&](const Item* u) {
        int64_t l = 0;
        for (int w = 0; w < U; ++w) l = std::max(l, item_work(u[w]));
        return l;
    };
    if (MF_WIDE_XCD) {
        // Runs of workgroups on one key range, most work first, are dealt
        // to the queue with the least work so far; each queue then runs its
        // workgroups most work first, and the queues are interleaved.
        constexpr int X = 8;
        const size_t nu = wunits.size();
        std::vector<int64_t> work(nu);
        for (size_t i = 0; i < nu; ++i) work[i] = unit_work(wunits[i]);
        auto same_range = [&](size_t x, size_t y) {
            const Item& a = wunits[x][0];
            const Item& b = wunits[y][0];
            // one key range; in a mixed plan one (sequence, kv head), whose
            // quads' ranges overlap
            return a[0] == b[0] && a[1] == b[1] && (mixed || device || (a[4] == b[4] && a[5] == b[5]));
        };
        // run r holds units [run_begin[r], run_begin[r + 1])
        std::vector<size_t> run_begin;
        std::vector<int64_t> run_work;
        for (size_t i = 0; i < nu; ++i) {
            if (i >= shared_items.size() / U || run_begin.empty() || !same_range(i - 1, i)) {
                run_begin.push_back(i);
                run_work.push_back(0);
            }
            run_work.back() += work[i];
        }
        const size_t nruns = run_begin.size();
        run_begin.push_back(nu);
        std::vector<size_t> order(nruns);
        for (size_t i = 0; i < nruns; ++i) order[i] = i;
        std::stable_sort(order.begin(), order.end(), [&](size_t x, size_t y) { return run_work[x] > run_work[y]; });
        // queue x holds exactly the workgroups at wide positions x mod 8; a
        // run that no queue has room for is split over the roomiest ones
        std::vector<size_t> queue[X];
        int64_t load[X] = {};
        for (auto& q : queue) q.reserve(nu / X + 1);
        auto room = [&](int x) { return (int64_t)(nu / X + (x < (int)(nu % X) ? 1 : 0)) - (int64_t)queue[x].size(); };
        for (size_t ri : order) {
            size_t i = run_begin[ri];
            const size_t end = run_begin[ri + 1];
            while (i < end) {
                int best = -1;
                for (int x = 0; x < X; ++x)
                    if (room(x) >= (int64_t)(end - i) && (best < 0 || load[x] < load[best])) best = x;
                if (best < 0) {
                    for (int x = 0; x < X; ++x)
                        if (best < 0 || room(x) > room(best)) best = x;
                }
                const size_t take = std::min<size_t>(end - i, (size_t)room(best));
                for (size_t t = 0; t < take; ++t, ++i) {
                    queue[best].push_back(i);
                    load[best] += work[i];
                }
            }
        }
        for (auto& q : queue)
            std::stable_sort(q.begin(), q.end(), [&](size_t x, size_t y) { return work[x] > work[y]; });
        int64_t wi = n_narrow;
        for (size_t k = 0;; ++k) {
            bool any = false;
            for (int x = 0; x < X; ++x) {
                if (k >= queue[x].size()) continue;
                any = true;
                const Item* u = wunits[queue[x][k]];
                for (int w = 0; w < U; ++w, ++wi) std::copy(u[w].begin(), u[w].end(), items + wi * MF_PLAN_ITEM_INTS);
            }
            if (!any) break;
        }
    } else {
        emit(wunits, n_narrow);
    }
    return MF_OK;
}
}  // namespace

extern "C" int mf_attention_plan(int num_seqs, const int32_t* cu_seqlens, const int32_t* kv_lens,
                                 int num_q_heads, int num_kv_heads, int head_dim, int dtype,
                                 int partition_tiles, int32_t* items, int64_t items_capacity,
                                 int32_t* merges, int64_t merges_capacity, int64_t* counts) {
    return attention_plan(num_seqs, cu_seqlens, kv_lens, num_q_heads, num_kv_heads, head_dim, dtype,
                          partition_tiles, 0, true, items, items_capacity, merges, merges_capacity, counts);
}

extern "C" int mf_attention_plan_device(int num_seqs, const int32_t* cu_seqlens, const int32_t* kv_lens,
                                        int num_q_heads, int num_kv_heads, int head_dim, int dtype, int num_cus,
                                        int32_t* items, int64_t items_capacity, int32_t* merges,
                                        int64_t merges_capacity, int64_t* counts) {
    if (num_cus <= 0) return MF_ERR_ARG;
    return attention_plan(num_seqs, cu_seqlens, kv_lens, num_q_heads, num_kv_heads, head_dim, dtype, 0, num_cus, true,
                          items, items_capacity, merges, merges_capacity, counts);
}

extern "C" int mf_attention_plan_merge_free(int num_seqs, const int32_t* cu_seqlens, const int32_t* kv_lens,
                                            int num_q_heads, int num_kv_heads, int head_dim, int dtype,
                                            int num_cus, int32_t* items, int64_t items_capacity, int32_t* merges,
                                            int64_t merges_capacity, int64_t* counts) {
    if (num_cus <= 0) return MF_ERR_ARG;
    return attention_plan(num_seqs, cu_seqlens, kv_lens, num_q_heads, num_kv_heads, head_dim, dtype, 0, num_cus, false,
                          items, items_capacity, merges, merges_capacity, counts);
}

// Slice plan for a large decode launch (attn_slice_kernel). The sequences'
// 16-key tiles, in sequence order, are cut into slices of about
// total / (num_cus * MF_SLICE_WAVES_PER_CU / Hkv) tiles, so one wave per
// (slice, kv head) fills the GPU exactly once at one workgroup per CU. A slice holds at most MF_SLICE_MAX_SEGMENTS
// segments and MF_SLICE_MAX_TILES tiles once each segment is padded to a
// multiple of the kernel's ring depth; a workload whose even share would
// exceed that gets more slices (a second round). A sequence cut across
// slices leaves one partial per piece and kv head, merged afterwards.
extern "C" int mf_attention_plan_slices(int num_seqs, const int32_t* cu_seqlens, const int32_t* kv_lens,
                                        int num_q_heads, int num_kv_heads, int head_dim, int dtype,
                                        int num_cus, int min_tiles_per_wave, int32_t* slices,
                                        int64_t slices_capacity, int32_t* merges, int64_t merges_capacity,
                                        int64_t* counts) {
    if (num_seqs < 0 || num_q_heads <= 0 || num_kv_heads <= 0 || head_dim <= 0 || !counts || num_cus <= 0 ||
        min_tiles_per_wave < 0)
        return MF_ERR_ARG;
    const int64_t resident_waves = (int64_t)num_cus * MF_SLICE_WAVES_PER_CU;
    if (num_q_heads % num_kv_heads) return MF_ERR_ARG;
    if (num_seqs > 0 && (!cu_seqlens || !kv_lens)) return MF_ERR_ARG;
    const int DP = mf::padded_head_dim(dtype, head_dim);
    if (!mf::dtype_ok(dtype) || !DP) return MF_ERR_UNSUPPORTED;
    const int G = num_q_heads / num_kv_heads;
    const int Hkv = num_kv_heads;
    counts[0] = counts[1] = counts[2] = counts[3] = 0;
    // Decode only: one query row per sequence, whose heads fit one column
    // tile, and head_dim at one of the kernel's sizes.
    if (DP != head_dim || G > 16) return MF_ERR_UNSUPPORTED;
    int64_t total = 0;
    for (int s = 0; s < num_seqs; ++s) {
        const int qlen = cu_seqlens[s + 1] - cu_seqlens[s];
        if (qlen < 0) return MF_ERR_ARG;
        if (kv_lens[s] <= 0 || qlen == 0) continue;
        if (qlen != 1) return MF_ERR_UNSUPPORTED;
        total += (kv_lens[s] + 15) / 16;
    }
    // Launches whose tiles give each resident wave fewer than
    // min_tiles_per_wave get no slice plan (counts stay zero): at
    // MF_SLICE_MIN_TILES and below, per-range items fit them in one round.
    if (total == 0 || total * Hkv < (int64_t)min_tiles_per_wave * resident_waves) return MF_OK;

    // Slices per round fill the GPU once; a workload whose even share would
    // not fit one slice runs whole rounds of equal slices (a round with only
    // a few slices would leave the GPU idle for its whole length). A slice's
    // real tiles stay below MF_SLICE_MAX_TILES by enough for the padding of
    // sixteen segments, so padding rarely closes a slice early.
    constexpr int NB = MF_NARROW_DEPTH;
    const int64_t base_slices = std::max<int64_t>(1, resident_waves / Hkv);
    const int64_t fill_cap = mf::kSliceMaxTiles - 16 * (NB - 1);
    const int64_t rounds = (total + base_slices * fill_cap - 1) / (base_slices * fill_cap);
    const int64_t want = rounds * base_slices;
    // slice i carries total / want tiles, one more for the first total % want
    const int64_t share = total / want, extra = total % want;

    // First walk: cut the slices (segment = sequence, kt0, kt1).
    struct Seg { int s, kt0, kt1; };
    std::vector<Seg> segs;
    std::vector<int64_t> begins;  // first segment of each slice
    std::vector<int> padded;      // padded tiles of each slice
    int64_t cur_real = 0, target = 0;
    int cur_pad = 0, cur_n = 0;
    auto open_slice = [&]() {
        target = std::max<int64_t>(1, share + ((int64_t)begins.size() < extra ? 1 : 0));
        begins.push_back((int64_t)segs.size());
        padded.push_back(0);
        cur_real = 0;
        cur_pad = 0;
        cur_n = 0;
    };
    open_slice();
    for (int s = 0; s < num_seqs; ++s) {
        const int qlen = cu_seqlens[s + 1] - cu_seqlens[s];
        if (kv_lens[s] <= 0 || qlen == 0) continue;
        const int T = (kv_lens[s] + 15) / 16;
        int kt = 0;
        while (kt < T) {
            const int64_t room_pad = mf::kSliceMaxTiles - cur_pad;
            if (cur_n == mf::kSliceMaxSegments || cur_real >= target || room_pad < NB) {
                open_slice();
                continue;
            }
            const int64_t take = std::min<int64_t>({(int64_t)(T - kt), target - cur_real, room_pad / NB * NB});
            segs.push_back({s, kt, (int)(kt + take)});
            cur_real += take;
            cur_pad += (int)((take + NB - 1) / NB * NB);
            padded.back() = cur_pad;
            ++cur_n;
            kt += (int)take;
        }
    }
    if (padded.back() == 0) {  // a slice opened after the last segment
        begins.pop_back();
        padded.pop_back();
    }
    const int64_t n_slices = (int64_t)begins.size();
    const int64_t n_segs = (int64_t)segs.size();

    // Pieces per sequence: slot ranges and merge records for split ones.
    std::vector<int> pieces(num_seqs, 0);
    for (const Seg& g : segs) ++pieces[g.s];
    int64_t n_merges = 0, n_slots = 0;
    for (int s = 0; s < num_seqs; ++s)
        if (pieces[s] > 1) {
            n_merges += Hkv;
            n_slots += (int64_t)Hkv * pieces[s];
        }
    counts[0] = n_slices;
    counts[1] = n_segs;
    counts[2] = n_merges;
    counts[3] = n_slots * 16 * (int64_t)(mf::part_dstride_for(head_dim) + 2);
    if (n_slices + n_segs > slices_capacity || n_merges > merges_capacity) return MF_ERR_WORKSPACE;
    if (!slices || (n_merges > 0 && !merges)) return MF_ERR_ARG;

    constexpr int R = MF_SLICE_INTS;
    for (int64_t i = 0; i < n_slices; ++i) {
        int32_t* o = slices + i * R;
        const int64_t end = i + 1 < n_slices ? begins[i + 1] : n_segs;
        std::fill(o, o + R, 0);
        o[0] = (int32_t)begins[i];
        o[1] = (int32_t)(end - begins[i]);
        o[2] = padded[i];
    }
    std::vector<int64_t> slot0(num_seqs, -1);
    int64_t slots = 0, wm = 0;
    for (int s = 0; s < num_seqs; ++s) {
        if (pieces[s] <= 1) continue;
        slot0[s] = slots;
        for (int h = 0; h < Hkv; ++h) {
            int32_t* o = merges + (wm++) * MF_PLAN_MERGE_INTS;
            o[0] = s;
            o[1] = h;
            o[2] = 0;
            o[3] = pieces[s];
            o[4] = (int32_t)(slots + (int64_t)h * pieces[s]);
            o[5] = 1;
            o[6] = cu_seqlens[s];
            o[7] = 1;
        }
        slots += (int64_t)Hkv * pieces[s];
    }
    std::vector<int> part(num_seqs, 0);
    for (int64_t i = 0; i < n_segs; ++i) {
        const Seg& g = segs[i];
        int32_t* o = slices + (n_slices + i) * R;
        o[0] = g.s;
        o[1] = g.kt0;
        o[2] = g.kt1;
        o[3] = cu_seqlens[g.s];
        o[4] = kv_lens[g.s];
        o[5] = (int32_t)slot0[g.s];
        o[6] = pieces[g.s];
        o[7] = part[g.s]++;
    }
    return MF_OK;
}

namespace {
int paged_attention_impl(
    const void* q, int64_t q_stride_row, int64_t q_stride_head, void* out, int64_t out_stride_row,
    int64_t out_stride_head, int dtype, const void* k_pool, const void* v_pool,
    int64_t pool_stride_block, int64_t pool_stride_slot, int64_t pool_stride_head, int block_size,
    const int32_t* block_tables, int64_t block_table_stride, const int32_t* cu_seqlens,
    const int32_t* kv_lens, const int64_t* positions, const int32_t* row_map,
    const int32_t* pool_lens, const void* new_k, const void* new_v, int64_t new_stride_row,
    int64_t new_stride_head, int num_q_heads, int num_kv_heads, int head_dim, float scale,
    const int32_t* plan_items, int64_t num_items_narrow, int64_t num_items_wide,
    const int32_t* plan_merges, int64_t num_merges, float* partials, int64_t partials_floats,
    int32_t* merge_counters, const int32_t* device_counts, mf_stream_t stream, bool sliced = false,
    const int64_t* write_slots = nullptr, int64_t write_rows = 0, int64_t write_num_slots = 0,
    bool tail_inflight = false) {
    using namespace mf;
    if (!(std::fabs(scale) < INFINITY)) return MF_ERR_ARG;  // NaN or infinite
    if (!dtype_ok(dtype) || num_q_heads <= 0 || num_kv_heads <= 0 || num_q_heads % num_kv_heads ||
        block_size <= 0 || num_items_narrow < 0 || num_items_wide < 0 || num_merges < 0)
        return MF_ERR_ARG;
    const int DP = padded_head_dim(dtype, head_dim);
    if (!DP) return MF_ERR_UNSUPPORTED;
    // A call may carry only items (partials left for a later merge-only call)
    // or only merges; both are how a caller times the two kernels apart.
    if (num_items_narrow + num_items_wide == 0 && num_merges == 0 && write_rows == 0) return MF_OK;
    if (!q || !out || !k_pool || !v_pool || !block_tables || !cu_seqlens || !kv_lens || !positions)
        return MF_ERR_ARG;
    if (num_items_narrow + num_items_wide > 0 && !plan_items) return MF_ERR_ARG;
    // Range-plan items run in workgroups of four and a wave loads its item
    // before its count check: both counts are whole workgroups, as plans make
    // them (a slice plan's counts are slices and segments).
    if (!sliced && ((num_items_narrow % kWaves) || (num_items_wide % kWaves))) return MF_ERR_ARG;
    if (pool_lens && (!new_k || !new_v)) return MF_ERR_ARG;
    if (num_merges > 0 && (!plan_merges || !partials || partials_floats <= 0)) return MF_ERR_WORKSPACE;
    // 16-byte row loads need 16-byte aligned rows.
    const int es = dtype_size(dtype);
    const int64_t epl = 16 / es;
    const int64_t strides[] = {q_stride_row, q_stride_head, pool_stride_block, pool_stride_slot,
                               pool_stride_head};
    for (int64_t st : strides)
        if (st % epl) return MF_ERR_ARG;
    if (((uintptr_t)q | (uintptr_t)k_pool | (uintptr_t)v_pool) & 15) return MF_ERR_ARG;
    if (pool_lens && ((new_stride_row % epl) || (new_stride_head % epl) ||
                      (((uintptr_t)new_k | (uintptr_t)new_v) & 15)))
        return MF_ERR_ARG;
    const int out_align = std::min(16, 4 * (DP / 16) * es);
    if ((out_stride_row * es) % out_align || (out_stride_head * es) % out_align ||
        ((uintptr_t)out % out_align))
        return MF_ERR_ARG;

    AttnArgs a{};
    a.q = (const char*)q;
    a.q_sr = q_stride_row;
    a.q_sh = q_stride_head;
    a.out = (char*)out;
    a.o_sr = out_stride_row;
    a.o_sh = out_stride_head;
    a.k_pool = (const char*)k_pool;
    a.v_pool = (const char*)v_pool;
    a.p_sb = pool_stride_block;
    a.p_ss = pool_stride_slot;
    a.p_sh = pool_stride_head;
    a.block_size = block_size;
    a.block_tables = block_tables;
    a.bt_stride = block_table_stride;
    a.cu_seqlens = cu_seqlens;
    a.kv_lens = kv_lens;
    a.positions = positions;
    a.row_map = row_map;
    a.pool_lens = pool_lens;
    a.new_k = (const char*)new_k;
    a.new_v = (const char*)new_v;
    a.n_sr = new_stride_row;
    a.n_sh = new_stride_head;
    a.G = num_q_heads / num_kv_heads;
    a.head_dim = head_dim;
    // Scores are scaled inside the exponent, which needs a positive factor:
    // a negative scale flips the sign of Q instead (exact), and a zero scale
    // becomes 2^-100, for which every 2^(s * scale - m) rounds to exactly 1,
    // the uniform weights a zero scale gives.
    a.q_sign = scale < 0.f ? (es == 4 ? 0x80000000u : 0x80008000u) : 0u;
    a.scale_log2 = scale == 0.f ? 0x1p-100f : std::fabs(scale) * 1.4426950408889634f;
    a.inv_scale_log2 = 1.f / a.scale_log2;
    a.partials = partials;
    a.part_dstride = part_dstride_for(head_dim);
    a.merges = plan_merges;
    a.counters = num_merges > 0 ? merge_counters : nullptr;
    a.num_kv_heads = num_kv_heads;
    const bool fast = block_size == 16 && head_dim == DP;
    hipStream_t st = (hipStream_t)stream;
    if (tail_inflight) {
        if (!new_k || !new_v || row_map || pool_lens || write_rows < 0 || write_num_slots < 0) return MF_ERR_ARG;
        if (write_rows > 0 && !write_slots) return MF_ERR_ARG;
        if ((new_stride_row % epl) || (new_stride_head % epl) || (((uintptr_t)new_k | (uintptr_t)new_v) & 15))
            return MF_ERR_ARG;
        if (!fast) {
            // other block sizes and padded head_dims: the write, then the
            // attention reading every key from the pool (same result, two launches)
            if (write_rows > 0) {
                if (int sw = mf_kv_write(new_k, new_v, dtype, new_stride_row, new_stride_head, write_slots,
                                         write_rows, const_cast<void*>(k_pool), const_cast<void*>(v_pool), dtype,
                                         pool_stride_block, pool_stride_slot, pool_stride_head, block_size,
                                         write_num_slots, num_kv_heads, head_dim, stream))
                    return sw;
            }
            tail_inflight = false;
        } else {
            // the copy: 16-byte pieces of every new row's K and V, about four
            // per thread of the copy workgroups
            const int64_t pieces = write_rows * 2 * num_kv_heads * (head_dim * es / 16);
            if (pieces > INT_MAX / 2) return MF_ERR_ARG;
            a.w_slots = write_slots;
            a.w_rows = (int)write_rows;
            a.w_num_slots = write_num_slots;
            a.w_blocks = pieces > 0 ? (int)std::min<int64_t>(1024, (pieces + 1023) / 1024) : 0;
        }
    }

    if (sliced && (!fast || row_map || pool_lens || merge_counters || device_counts || tail_inflight))
        return MF_ERR_UNSUPPORTED;
#define MF_ATTN_CASE(DT, DPV)                                                                  \
    if (dtype == DT && DP == DPV)                                                              \
        return sliced ? launch_slices<DT, DPV>(a, plan_items, num_items_narrow, num_kv_heads,  \
                                               plan_merges, num_merges, st)                    \
                      : (tail_inflight ? launch_attention<DT, DPV, true>(a, plan_items, num_items_narrow, \
                                                                         num_items_wide, plan_merges, num_merges, \
                                                                         fast, device_counts, st) \
                                       : launch_attention<DT, DPV>(a, plan_items, num_items_narrow, num_items_wide, \
                                                                   plan_merges, num_merges, fast, device_counts, st));
    MF_ATTN_CASE(MF_F32, 16)
    MF_ATTN_CASE(MF_F32, 32)
    MF_ATTN_CASE(MF_F32, 64)
    MF_ATTN_CASE(MF_F32, 128)
    MF_ATTN_CASE(MF_BF16, 32)
    MF_ATTN_CASE(MF_BF16, 64)
    MF_ATTN_CASE(MF_BF16, 128)
    MF_ATTN_CASE(MF_BF16, 256)
    MF_ATTN_CASE(MF_F16, 32)
    MF_ATTN_CASE(MF_F16, 64)
    MF_ATTN_CASE(MF_F16, 128)
    MF_ATTN_CASE(MF_F16, 256)
#undef MF_ATTN_CASE
    return MF_ERR_UNSUPPORTED;
}
}  // namespace

extern "C" int mf_paged_attention(
    const void* q, int64_t q_stride_row, int64_t q_stride_head, void* out, int64_t out_stride_row,
    int64_t out_stride_head, int dtype, const void* k_pool, const void* v_pool,
    int64_t pool_stride_block, int64_t pool_stride_slot, int64_t pool_stride_head, int block_size,
    const int32_t* block_tables, int64_t block_table_stride, const int32_t* cu_seqlens,
    const int32_t* kv_lens, const int64_t* positions, const int32_t* row_map,
    const int32_t* pool_lens, const void* new_k, const void* new_v, int64_t new_stride_row,
    int64_t new_stride_head, int num_q_heads, int num_kv_heads, int head_dim, float scale,
    const int32_t* plan_items, int64_t num_items_narrow, int64_t num_items_wide,
    const int32_t* plan_merges, int64_t num_merges, float* partials, int64_t partials_floats,
    int32_t* merge_counters, mf_stream_t stream) {
    return paged_attention_impl(q, q_stride_row, q_stride_head, out, out_stride_row, out_stride_head, dtype,
                                k_pool, v_pool, pool_stride_block, pool_stride_slot, pool_stride_head,
                                block_size, block_tables, block_table_stride, cu_seqlens, kv_lens, positions,
                                row_map, pool_lens, new_k, new_v, new_stride_row, new_stride_head, num_q_heads,
                                num_kv_heads, head_dim, scale, plan_items, num_items_narrow, num_items_wide,
                                plan_merges, num_merges, partials, partials_floats, merge_counters, nullptr,
                                stream);
}

extern "C" int mf_paged_attention_slices(
    const void* q, int64_t q_stride_row, int64_t q_stride_head, void* out, int64_t out_stride_row,
    int64_t out_stride_head, int dtype, const void* k_pool, const void* v_pool,
    int64_t pool_stride_block, int64_t pool_stride_slot, int64_t pool_stride_head, int block_size,
    const int32_t* block_tables, int64_t block_table_stride, const int32_t* cu_seqlens,
    const int32_t* kv_lens, const int64_t* positions, int num_q_heads, int num_kv_heads, int head_dim,
    float scale, const int32_t* slices, int64_t num_slices, int64_t num_segments,
    const int32_t* plan_merges, int64_t num_merges, float* partials, int64_t partials_floats,
    mf_stream_t stream) {
    return paged_attention_impl(q, q_stride_row, q_stride_head, out, out_stride_row, out_stride_head, dtype,
                                k_pool, v_pool, pool_stride_block, pool_stride_slot, pool_stride_head,
                                block_size, block_tables, block_table_stride, cu_seqlens, kv_lens, positions,
                                nullptr, nullptr, nullptr, nullptr, 0, 0, num_q_heads, num_kv_heads, head_dim,
                                scale, slices, num_slices, num_segments, plan_merges, num_merges, partials,
                                partials_floats, nullptr, nullptr, stream, /*sliced=*/true);
}

extern "C" int mf_paged_attention_counted(
    const void* q, int64_t q_stride_row, int64_t q_stride_head, void* out, int64_t out_stride_row,
    int64_t out_stride_head, int dtype, const void* k_pool, const void* v_pool,
    int64_t pool_stride_block, int64_t pool_stride_slot, int64_t pool_stride_head, int block_size,
    const int32_t* block_tables, int64_t block_table_stride, const int32_t* cu_seqlens,
    const int32_t* kv_lens, const int64_t* positions, const int32_t* row_map,
    const int32_t* pool_lens, const void* new_k, const void* new_v, int64_t new_stride_row,
    int64_t new_stride_head, int num_q_heads, int num_kv_heads, int head_dim, float scale,
    const int32_t* plan_items, int64_t capacity_narrow, int64_t capacity_wide,
    const int32_t* plan_merges, int64_t capacity_merges, const int32_t* device_counts, float* partials,
    int64_t partials_floats, mf_stream_t stream) {
    if (!device_counts) return MF_ERR_ARG;
    return paged_attention_impl(q, q_stride_row, q_stride_head, out, out_stride_row, out_stride_head, dtype,
                                k_pool, v_pool, pool_stride_block, pool_stride_slot, pool_stride_head,
                                block_size, block_tables, block_table_stride, cu_seqlens, kv_lens, positions,
                                row_map, pool_lens, new_k, new_v, new_stride_row, new_stride_head, num_q_heads,
                                num_kv_heads, head_dim, scale, plan_items, capacity_narrow, capacity_wide,
                                plan_merges, capacity_merges, partials, partials_floats, nullptr,
                                device_counts, stream);
}

extern "C" int mf_paged_attention_kv_write(
    const void* q, int64_t q_stride_row, int64_t q_stride_head, void* out, int64_t out_stride_row,
    int64_t out_stride_head, int dtype, void* k_pool, void* v_pool, int64_t pool_stride_block,
    int64_t pool_stride_slot, int64_t pool_stride_head, int block_size, const int32_t* block_tables,
    int64_t block_table_stride, const int32_t* cu_seqlens, const int32_t* kv_lens, const int64_t* positions,
    const void* new_k, const void* new_v, int64_t new_stride_row, int64_t new_stride_head,
    const int64_t* slot_mapping, int64_t num_new_rows, int64_t num_slots, int num_q_heads, int num_kv_heads,
    int head_dim, float scale, const int32_t* plan_items, int64_t num_items_narrow, int64_t num_items_wide,
    const int32_t* plan_merges, int64_t num_merges, const int32_t* device_counts, float* partials,
    int64_t partials_floats, mf_stream_t stream) {
    return paged_attention_impl(q, q_stride_row, q_stride_head, out, out_stride_row, out_stride_head, dtype,
                                k_pool, v_pool, pool_stride_block, pool_stride_slot, pool_stride_head,
                                block_size, block_tables, block_table_stride, cu_seqlens, kv_lens, positions,
                                nullptr, nullptr, new_k, new_v, new_stride_row, new_stride_head, num_q_heads,
                                num_kv_heads, head_dim, scale, plan_items, num_items_narrow, num_items_wide,
                                plan_merges, num_merges, partials, partials_floats, nullptr, device_counts,
                                stream, /*sliced=*/false, slot_mapping, num_new_rows, num_slots,
                                /*tail_inflight=*/true);
}

// ------------------------------------------------------- no-allocation entry
//
// mf_paged_attention for callers that cannot allocate device memory: the
// split-K partials go to `scratch`, a library-owned device array that every
// GPU holding this code object keeps until the process ends. In host code the
// array's name is only a stand-in for the symbol; its device address, which
// differs per GPU, comes from hipGetSymbolAddress on the first call on each
// device and is the only form host code ever passes to a kernel. Nothing in
// it needs clearing between calls (every partial slot is written before the
// merge reads it), and calls that overlap on one GPU race on it.
static __device__ __align__(256) float scratch[MF_NOALLOC_PARTIALS_FLOATS];

namespace {
constexpr int kMaxScratchDevices = 64;
std::atomic<float*> g_scratch_ptr[kMaxScratchDevices];
std::mutex g_scratch_mu;

// Device address of the current device's `scratch`, looked up once per device.
int scratch_for_current_device(float** out) {
    int dev = -1;
    hipError_t err = hipGetDevice(&dev);
    if (err != hipSuccess) {
        mf::set_last_hip_error((int)err);
        return MF_ERR_HIP;
    }
    if (dev < 0 || dev >= kMaxScratchDevices) return MF_ERR_UNSUPPORTED;
    float* p = g_scratch_ptr[dev].load(std::memory_order_acquire);
    if (!p) {
        std::lock_guard<std::mutex> lock(g_scratch_mu);
        p = g_scratch_ptr[dev].load(std::memory_order_relaxed);
        if (!p) {
            void* addr = nullptr;
            err = hipGetSymbolAddress(&addr, HIP_SYMBOL(scratch));
            if (err != hipSuccess || !addr) {
                mf::set_last_hip_error((int)err);
                return MF_ERR_HIP;
            }
            p = (float*)addr;
            g_scratch_ptr[dev].store(p, std::memory_order_release);
        }
    }
    *out = p;
    return MF_OK;
}
}  // namespace

extern "C" int mf_paged_attention_noalloc(
    const void* q, int64_t q_stride_row, int64_t q_stride_head, void* out, int64_t out_stride_row,
    int64_t out_stride_head, int dtype, const void* k_pool, const void* v_pool,
    int64_t pool_stride_block, int64_t pool_stride_slot, int64_t pool_stride_head, int block_size,
    const int32_t* block_tables, int64_t block_table_stride, const int32_t* cu_seqlens,
    const int32_t* kv_lens, const int64_t* positions, const int32_t* row_map,
    const int32_t* pool_lens, const void* new_k, const void* new_v, int64_t new_stride_row,
    int64_t new_stride_head, int num_q_heads, int num_kv_heads, int head_dim, float scale,
    const int32_t* plan_items, int64_t num_items_narrow, int64_t num_items_wide,
    const int32_t* plan_merges, int64_t num_merges, int64_t partials_floats, mf_stream_t stream) {
    // sizes first: a plan that needs more than the array is refused before
    // anything touches the device
    if (partials_floats < 0) return MF_ERR_ARG;
    if (partials_floats > MF_NOALLOC_PARTIALS_FLOATS) return MF_ERR_WORKSPACE;
    float* partials = nullptr;
    if (int st = scratch_for_current_device(&partials)) return st;
    return paged_attention_impl(q, q_stride_row, q_stride_head, out, out_stride_row, out_stride_head, dtype,
                                k_pool, v_pool, pool_stride_block, pool_stride_slot, pool_stride_head,
                                block_size, block_tables, block_table_stride, cu_seqlens, kv_lens, positions,
                                row_map, pool_lens, new_k, new_v, new_stride_row, new_stride_head, num_q_heads,
                                num_kv_heads, head_dim, scale, plan_items, num_items_narrow, num_items_wide,
                                plan_merges, num_merges, partials, MF_NOALLOC_PARTIALS_FLOATS, nullptr,
                                nullptr, stream);
}

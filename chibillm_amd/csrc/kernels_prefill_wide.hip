// Chunked-prefill causal attention over paged KV of 256-wide heads with MFMA
// tiles (gfx950), bf16 and fp16. The maths, the operand layouts and the hand-over
// of split tiles are those of kernels_prefill.hip; what differs follows from the
// head's width.
//
// One workgroup of four waves, one per SIMD with up to 512 registers a lane
// (an O^T of 256 features by 32 queries alone takes 128, Q^T 64), owns 128 / G
// rows of a query tile for G <= 4 query heads of one kv head; a GQA group of 8
// takes two workgroups. Per 32-key block and wave: 16 v_mfma_f32_32x32x16 for
// S^T = K . Q^T and 48 for O^T += V^T . P^T, because P^T enters as three 16-bit
// terms, each the rounding of what those before it left: together all 24 bits
// of a probability's significand, which the decode kernels hold in 32 bits for
// such heads too. fp16 terms are taken at 2^6 times the probability, which the
// final division removes, so that what fp16's smallest value cuts off is at most
// 2^-31 of the largest probability, below the accumulators' own rounding.
// Over 26 batches of 1 to 4 sequences (1 to 4 kv heads, groups of 2 and 4, 2 to
// 512 rows over 0 to 700 tokens, N(0, 1)) the error against 64 bits is that of
// 32-bit probabilities (1.6e-3 to 1.9e-3 in bf16, 2.2e-4 to 2.4e-4 in fp16, the
// rounding of stored values; ratio 1.000004 in the mean, 0.99994 to 1.0002). Two
// terms, 16 bits in bf16, measured the same on these values (1.000005) and took
// 62.5 us for the launch below instead of 67.2; one gives 2.9e-3.
//
// With one wave on a SIMD nothing else hides a wait, so K operands are read a
// block ahead: iteration kb multiplies K(kb), already in registers, while the
// vector ALU forms the probabilities of block kb - 1 and V(kb - 1) is read;
// then O^T of block kb - 1 is multiplied while K(kb + 1) is read and the scores
// of block kb are masked and searched for maxima. K has to be staged one block
// sooner than V: K and V have four LDS stages each (132 KiB, one workgroup per
// compute unit), iteration kb loads K(kb + 3) and V(kb + 2), and its barrier
// publishes K(kb + 2) and V(kb).
//
// Four sequences of 300 to 512 rows behind 700 tokens (2 kv heads, 8 q heads,
// gated, 12.1 GFLOP) take 66.7 us with their two rotations, of them 61.6 here (in
// a kernel trace; the general path took 3,900 to 4,100): 104 workgroups of 32 rows, of which the
// eight that start a sequence, 23 key blocks each, are not cut (fewer than three ranges'
// worth of blocks) and the others have their 24 to 38 blocks in two ranges. The
// uncut ones are the longest chains, and what bounds the launch is such a chain, not
// the matrix cores. With two-term probabilities a block took 3,500 cycles of a wave:
// 1,000 to issue its loads (about 32 bytes a cycle and compute unit pass to LDS), 890
// for the scores and probabilities, 720 for P.V, 700 for maxima, waits and
// rescales; the third term adds about 480. Issuing the loads in twos between those
// phases took 64.1 to 64.7 us in all instead of 62.3; reading both halves of V
// before the scores 64.7.
#include "ckv_internal.h"
#include "prefill_records.h"
#include "prefill_tile.h"

#include <algorithm>
#include <cfloat>
#include <cstdlib>

namespace ckv {
namespace {

constexpr uint32_t dim = 256;
constexpr uint32_t page_tokens = 16;
constexpr uint32_t block_keys = 32;
constexpr uint32_t waves = 4;
constexpr uint32_t n_stages = 4;
constexpr uint32_t k_steps = dim / 16; // products of a block's S^T
constexpr uint32_t tiles_o = dim / 32; // accumulators of O^T

// K stage: the block's 32 key rows of 512 bytes in order, the 16-byte chunks of
// row k in the order chunk ^ (k % 16): a DMA instruction moves two whole rows
// (eight full cache lines), and the 16 lanes that read a chunk of 16 rows
// together find it at 16 different bank offsets (staged in operand order, 32 bytes
// of each of 32 rows per instruction, that launch took 62.9 us instead of
// 62.3, with its rotations and two-term probabilities).
constexpr uint32_t k_stage_bytes = block_keys * dim * 2;
// V stage: two halves of 128 features, each as kernels_prefill.hip stages a
// 128-wide head: 8 groups of 4 key rows, 64 bytes after each group.
constexpr uint32_t vg_bytes = 1024 + 64;
constexpr uint32_t v_half_bytes = 8 * vg_bytes;
constexpr uint32_t v_stage_bytes = 2 * v_half_bytes;
constexpr uint32_t regions = 4; // K regions, and V groups, a wave stages per block

// 16-bit terms of a probability.
constexpr int terms = 3;
// Scale of fp16 probabilities (log2): with the running maximum up to 2^8 stale
// they reach 2^14, within fp16's range.
constexpr float p_scale_f16 = 6.0f;

// The source of masked K and V rows.
__device__ const uint4 zero_row[32] = {};

template <bool F16>
__device__ __forceinline__ float word_value(uint32_t w, int e)
{
    if constexpr (F16)
        return half_value<true>(static_cast<uint16_t>(w >> (16 * e)));
    else
        return __builtin_bit_cast(float, e ? w & 0xFFFF0000u : w << 16);
}

__device__ __forceinline__ void wait_all_but(uint32_t loads)
{
    if (loads >= 12)
        __builtin_amdgcn_s_waitcnt(0x0F7C); // vmcnt(12)
    else if (loads >= 8)
        __builtin_amdgcn_s_waitcnt(0x0F78);
    else if (loads >= 4)
        __builtin_amdgcn_s_waitcnt(0x0F74);
    else
        __builtin_amdgcn_s_waitcnt(0x0F70);
}

// Sum over each row of 16 lanes, result in every lane of the row.
__device__ __forceinline__ float row16_sum(float v)
{
    auto add = [&](int moved) { v += __builtin_bit_cast(float, moved); };
    const auto bits = [&]() { return __builtin_bit_cast(int, v); };
    add(__builtin_amdgcn_mov_dpp(bits(), 0xB1, 0xF, 0xF, true));  // quad_perm [1,0,3,2]
    add(__builtin_amdgcn_mov_dpp(bits(), 0x4E, 0xF, 0xF, true));  // quad_perm [2,3,0,1]
    add(__builtin_amdgcn_mov_dpp(bits(), 0x141, 0xF, 0xF, true)); // row_half_mirror
    add(__builtin_amdgcn_mov_dpp(bits(), 0x140, 0xF, 0xF, true)); // row_mirror
    return v;
}

// Up to alone_queries rows of one query head (bits of `rows`, from row r0 on) against
// their keys by vector arithmetic: what a wave falls back to for the queries to
// which the tile gave a value that is not finite. A product with P^T
// multiplies every key of a block for all its queries, so an infinity or NaN
// in a V row also meets the zeros of the queries that do not attend it (and of a
// low term), and 0 * inf is NaN; the decode kernels give such a row only to the
// queries that attend it, and so does this. Sixteen lanes hold a row, four rows
// a step, the next step's in flight; finite results never come here. An infinity
// early in a shared prefix sends every query of a launch here, so a K/V row read
// and widened serves several queries: with one in the first page of each
// sequence the launch below takes 1.81 ms (two at a time 2.29, eight 1.96, one
// 5.84; the general path took 3.93 for these rows). The cost grows with the
// rows' positions, as theirs did.
constexpr uint32_t alone_queries = 4;

template <bool F16>
__device__ __forceinline__ void attend_alone(const uint16_t* __restrict__ keys,
                                             const uint16_t* __restrict__ values,
                                             const uint32_t* __restrict__ table, uint32_t F,
                                             uint32_t rows, uint32_t pos0, const uint16_t* q,
                                             size_t q_stride, float c, const uint16_t* gate,
                                             uint16_t* out, uint32_t lane)
{
    constexpr uint32_t each = dim / 16, Q = alone_queries;
    const uint32_t f = (lane & 15) * each, sub = lane >> 4;
    struct words {
        u32x4_t w[2];
    };
    auto load = [&](const uint16_t* at) {
        return words { { reinterpret_cast<const u32x4_t*>(at + f)[0],
                         reinterpret_cast<const u32x4_t*>(at + f)[1] } };
    };
    auto widen = [](const words& r, float (&x)[each]) {
#pragma unroll
        for (uint32_t i = 0; i < each; ++i)
            x[i] = word_value<F16>(r.w[i / 8][i / 2 % 4], i % 2);
    };
    auto weight = [&](float ms, float to) { return __builtin_amdgcn_exp2f((ms - to) * c); };
    // the rows (the first again in the places left over) and their states, which
    // start at the lowest finite maximum: without keys a state weighs 0 or holds 0
    uint32_t row[Q], count = 0;
    float qf[Q][each], acc[Q][each], m[Q], l[Q];
#pragma unroll
    for (uint32_t i = 0; i < Q; ++i) {
        row[i] = rows ? __builtin_ctz(rows) : row[0];
        count += rows != 0;
        rows &= rows - (rows != 0);
        widen(load(q + row[i] * q_stride), qf[i]);
        m[i] = -FLT_MAX;
        l[i] = 0.0f;
#pragma unroll
        for (uint32_t j = 0; j < each; ++j)
            acc[i][j] = 0.0f;
    }
    const uint32_t last = pos0 + row[count - 1]; // the rows ascend
    uint32_t page = table[0];
    auto at_key = [&](uint32_t key) { // in the page at hand; past the last key, that one
        return ((uint64_t)page * page_tokens + min(key, last) % page_tokens) * F;
    };
    words k_next = load(keys + at_key(sub)), v_next = load(values + at_key(sub));
#pragma unroll 1
    for (uint32_t key0 = 0; key0 <= last; key0 += 4) {
        const words k_now = k_next, v_now = v_next;
        const uint32_t key = key0 + sub, next = key0 + 4;
        if (next <= last) {
            if (next % page_tokens == 0)
                page = table[next / page_tokens];
            k_next = load(keys + at_key(next + sub));
            v_next = load(values + at_key(next + sub));
        }
        float x[each], s[Q];
        widen(k_now, x);
#pragma unroll
        for (uint32_t i = 0; i < Q; ++i) {
            s[i] = 0.0f;
#pragma unroll
            for (uint32_t j = 0; j < each; ++j)
                s[i] = __builtin_fmaf(qf[i][j], x[j], s[i]);
            s[i] = row16_sum(s[i]);
        }
        widen(v_now, x);
#pragma unroll
        for (uint32_t i = 0; i < Q; ++i)
            if (key <= pos0 + row[i]) {
                const float m_new = fmaxf(m[i], s[i]);
                const float keep = weight(m[i], m_new), w = weight(s[i], m_new);
                m[i] = m_new;
                l[i] = l[i] * keep + w;
#pragma unroll
                for (uint32_t j = 0; j < each; ++j)
                    acc[i][j] = acc[i][j] * keep + w * x[j];
            }
    }
#pragma unroll
    for (uint32_t i = 0; i < Q; ++i) {
#pragma unroll
        for (uint32_t d = 16; d < 64; d *= 2) {
            const float m_other = __shfl_xor(m[i], d), l_other = __shfl_xor(l[i], d);
            const float m_new = fmaxf(m[i], m_other);
            const float keep = weight(m[i], m_new), w = weight(m_other, m_new);
            m[i] = m_new;
            l[i] = l[i] * keep + l_other * w;
#pragma unroll
            for (uint32_t j = 0; j < each; ++j) {
                const float other = __shfl_xor(acc[i][j], d);
                acc[i][j] = acc[i][j] * keep + other * w;
            }
        }
        if (i >= count || sub)
            continue;
        const float inv = 1.0f / l[i];
        const size_t at = row[i] * q_stride + f;
#pragma unroll
        for (uint32_t j = 0; j < each; j += 2) {
            float y[2] = { acc[i][j] * inv, acc[i][j + 1] * inv };
            if (gate)
                for (int e = 0; e < 2; ++e)
                    y[e] *= sigmoid(half_value<F16>(gate[at + j + e]));
            *reinterpret_cast<uint32_t*>(out + at + j) = pack2<F16>(y[0], y[1]);
        }
    }
}

// FAR: a layer spans more than 4 GiB, so page offsets take 64 bits.
template <int G, bool F16, bool FAR>
__global__ __launch_bounds__(64 * waves, 1) void prefill_wide_kernel(
    pool_view p, meta_view md, uint32_t layer, const uint16_t* __restrict__ q,
    uint16_t* __restrict__ out, uint32_t q_heads, float c, const uint16_t* __restrict__ gate,
    prefill_split split_scratch)
{
    __shared__ __attribute__((aligned(16))) uint8_t lds[n_stages * (k_stage_bytes + v_stage_bytes)];
    constexpr uint32_t tile_rows = 32 * waves / G;
    constexpr uint32_t subs = prefill_tile_rows / tile_rows; // workgroups per (tile, head pass, kv head)

    const uint32_t kv_heads = p.kv_heads;
    const uint32_t group = q_heads / kv_heads;
    const uint32_t passes = group / G; // 1, or 2 for groups of 8
    const uint32_t kvh = blockIdx.x % kv_heads;
    const uint32_t pass = blockIdx.x / kv_heads % passes;
    // key ranges vary slowest, as in kernels_prefill.hip
    const uint32_t n_split = split_scratch.n_split;
    const uint32_t n_rest = md.n_tiles * subs;
    const uint32_t rest = blockIdx.x / (kv_heads * passes) % n_rest;
    const uint32_t part = blockIdx.x / (kv_heads * passes) / n_rest;
    const uint32_t sub = rest % subs;
    const uint32_t tile = rest / subs;
    const uint4 te = *reinterpret_cast<const uint4*>(md.tiles + tile_entry_words * tile);
    const uint32_t count = te.y;
    const uint32_t r0 = sub * tile_rows;
    if (r0 >= count)
        return;
    const uint32_t nrows = min(tile_rows, count - r0);
    const uint32_t row0 = te.x + r0;
    const uint32_t pos0 = te.z + r0;
    const uint32_t pos_last = pos0 + nrows - 1;
    const uint32_t* table = md.table + te.w;
    const uint32_t n_blocks = pos_last / block_keys + 1;
    const uint32_t n_parts = prefill_range_count(n_blocks, n_split, split_scratch.min_blocks);
    if (part >= n_parts)
        return;
    uint32_t kb_begin, kb_end;
    prefill_range_bounds(n_blocks, n_parts, part, kb_begin, kb_end);

    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t n = lane & 31, g = lane >> 5;
    const uint32_t F = p.features;
    const size_t q_stride = (size_t)q_heads * dim;

    // this wave's q-block: one query head, tile rows 32 * (wave / G) + n
    const uint32_t rb = wave / G;
    const uint32_t head = kvh * group + pass * G + wave % G;
    const uint32_t row = rb * 32 + n;
    const bool valid = row < nrows;
    const uint32_t qpos = pos0 + min(row, nrows - 1);
    const size_t qoff = (size_t)(row0 + min(row, nrows - 1)) * q_stride + (size_t)head * dim;
    const uint32_t pos_lo = pos0 + rb * 32; // the q-block's first position (scalar)

    // Q^T: features 16ks + 8g .. +7 of query n (lanes past the tile's rows hold its
    // last row again; their results are not written)
    u32x4_t qr[k_steps];
#pragma unroll
    for (uint32_t ks = 0; ks < k_steps; ++ks)
        qr[ks] = *reinterpret_cast<const u32x4_t*>(q + qoff + ks * 16 + g * 8);

    // Staging: the wave moves K row pairs 2 wave, 2 wave + 8 of each page of the
    // block and V groups wave, wave + 4 of each half (the block's first and
    // second page), one DMA each.
    const uint64_t page_bytes = (uint64_t)page_tokens * F * 2;
    const uint64_t base_elems = layer * p.layer_elems + (uint64_t)kvh * dim;
    const uint8_t* kbytes = uniform_ptr(reinterpret_cast<const uint8_t*>(
        static_cast<const uint16_t*>(p.keys) + base_elems));
    const uint8_t* vbytes = uniform_ptr(reinterpret_cast<const uint8_t*>(
        static_cast<const uint16_t*>(p.values) + base_elems));
    const uint8_t* zbytes = reinterpret_cast<const uint8_t*>(zero_row);
    uint32_t k_row[2], k_off[2]; // this lane's key of a page and its source bytes there
#pragma unroll
    for (uint32_t i = 0; i < 2; ++i) {
        k_row[i] = 2 * wave + 8 * i + g;
        k_off[i] = k_row[i] * F * 2 + (n ^ k_row[i]) * 16;
    }
    const uint32_t v_key = 4 * (lane >> 4) + wave; // in either page
    const uint32_t v_off = (v_key * F + (lane & 15) * 8) * 2;
    const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds;
    auto k_stage = [&](uint32_t kb) { return kb % n_stages * k_stage_bytes; };
    auto v_stage = [&](uint32_t kb) {
        return n_stages * k_stage_bytes + kb % n_stages * v_stage_bytes;
    };

    const uint32_t last_entry = pos_last / page_tokens;
    using c32 = const __attribute__((address_space(4))) uint32_t;
    const auto* table_s = (const __attribute__((address_space(4))) uint8_t*)(uintptr_t)table;
    auto page_of = [&](uint32_t entry) { // a scalar load; past the tile's end, its last page
        return *(c32*)(table_s + 4 * (uint64_t)min(entry, last_entry));
    };
    auto page_at = [&](uint32_t page) { // a page's bytes from the layer's base
        return FAR ? page * page_bytes : (uint64_t)(page * (uint32_t)page_bytes);
    };
    auto load_k = [&](uint32_t kb, uint32_t pg0, uint32_t pg1) {
        const uint32_t key0 = kb * block_keys;
        const bool whole = key0 + block_keys - 1 <= pos_last;
#pragma unroll
        for (uint32_t r = 0; r < regions; ++r) { // the block's page r / 2, rows 8 * (r % 2) ..
            const uint32_t st = lds_base + k_stage(kb) + (wave + 4 * r) * 1024;
            const uint8_t* pk = kbytes + page_at(r / 2 ? pg1 : pg0);
            if (whole) {
                dma16_s(pk, k_off[r % 2], st);
            } else {
                const bool live = key0 + page_tokens * (r / 2) + k_row[r % 2] <= pos_last;
                dma16(live ? pk + k_off[r % 2] : zbytes + n * 16, st);
            }
        }
    };
    auto load_v = [&](uint32_t kb, uint32_t pg0, uint32_t pg1) {
        const uint32_t key0 = kb * block_keys;
        const bool whole = key0 + block_keys - 1 <= pos_last;
#pragma unroll
        for (uint32_t r = 0; r < regions; ++r) { // half r / 2, the block's page r % 2
            const uint32_t st = lds_base + v_stage(kb) + (r / 2) * v_half_bytes
                + (wave + 4 * (r % 2)) * vg_bytes;
            const uint8_t* pv = vbytes + page_at(r % 2 ? pg1 : pg0) + 256 * (r / 2);
            if (whole) {
                dma16_s(pv, v_off, st);
            } else {
                const bool live = key0 + page_tokens * (r % 2) + v_key <= pos_last;
                dma16(live ? pv + v_off : zbytes + (lane & 15) * 16, st);
            }
        }
    };

    f32x16_t o[tiles_o];
#pragma unroll
    for (uint32_t mt = 0; mt < tiles_o; ++mt)
        o[mt] = f32x16_t {};
    float m = -__builtin_inff(), l = 0.0f;
    float m_limit = -__builtin_inff();
    const float rescale_raw = rescale_log2 / c;
    f32x16_t sp; // scores of the block whose probabilities come next
    float mx = 0.0f;
    uint4 ka[k_steps];

    // A operand of step ks: chunk 2ks + g of key row key_row(n)
    const uint32_t kr_row = key_row(n) * (dim * 2), kr_swap = ((key_row(n) & 15) ^ g) * 16;
    auto read_k = [&](uint32_t kb) {
        const uint32_t base = lds_base + k_stage(kb) + kr_row;
#pragma unroll
        for (uint32_t ks = 0; ks < k_steps; ++ks) {
            const uint32_t at = base + (kr_swap ^ (32 * (ks % 8))); // chunk bit 4 is not swapped
            ka[ks] = __builtin_bit_cast(uint4, *(const __attribute__((address_space(3))) u32x4_t*)(uintptr_t)(at + 256 * (ks / 8)));
        }
    };
    const uint32_t vr_off = ((lane & 15) >> 2) * vg_bytes + (lane >> 5) * 512
        + ((lane >> 4) & 1) * 32 + (lane & 3) * 8;
    // A operands of O^T's accumulators 4 * half + mt (features 32mt + n of that
    // half of the head), keys 16h + 8g + 0..7
    auto read_v = [&](uint32_t kb, uint32_t half, uint4 (&va)[4][2]) {
        uint32_t vaddr = lds_base + v_stage(kb) + half * v_half_bytes + vr_off;
        asm volatile("" : "+v"(vaddr));
        auto* vb = (__attribute__((address_space(3))) uint8_t*)(uintptr_t)vaddr;
#pragma unroll
        for (uint32_t mt = 0; mt < 4; ++mt)
#pragma unroll
            for (uint32_t h = 0; h < 2; ++h) {
                auto* at = vb + 4 * h * vg_bytes + 64 * mt;
                const i16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (__attribute__((address_space(3))) i16x4_t*)at);
                const i16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (__attribute__((address_space(3))) i16x4_t*)(at + 256));
                const uint2 l2 = __builtin_bit_cast(uint2, lo), h2 = __builtin_bit_cast(uint2, hi);
                va[mt][h] = make_uint4(l2.x, l2.y, h2.x, h2.y);
            }
    };
    // the probabilities of sp as 16-bit terms, and their share of the denominator
    auto probabilities = [&](uint4 (&pt)[terms][2]) {
        // a range of the keys may hold none a query attends yet (m = -inf)
        const float bias = F16 ? p_scale_f16 : 0.0f;
        const float mc = m == -__builtin_inff() ? 0.0f : __builtin_fmaf(m, c, -bias);
#pragma unroll
        for (int r = 0; r < 16; ++r)
            sp[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(sp[r], c, -mc));
        float q4[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            q4[i] = (sp[4 * i] + sp[4 * i + 1]) + (sp[4 * i + 2] + sp[4 * i + 3]);
        l += (q4[0] + q4[1]) + (q4[2] + q4[3]);
        // each term the rounding of what the terms before it left
#pragma unroll
        for (int t = 0; t < terms; ++t) {
            uint32_t w[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                w[i] = pack2<F16>(sp[2 * i], sp[2 * i + 1]);
                if (t + 1 < terms) {
                    sp[2 * i] -= word_value<F16>(w[i], 0);
                    sp[2 * i + 1] -= word_value<F16>(w[i], 1);
                }
            }
#pragma unroll
            for (int h = 0; h < 2; ++h)
                pt[t][h] = make_uint4(w[4 * h], w[4 * h + 1], w[4 * h + 2], w[4 * h + 3]);
        }
    };
    auto qk = [&]() {
        f32x16_t s = {};
#pragma unroll
        for (uint32_t ks = 0; ks < k_steps; ++ks)
            s = mfma<F16>(ka[ks], __builtin_bit_cast(uint4, qr[ks]), s);
        asm volatile("" : "+v"(s)); // the vector ALU reads it next
        return s;
    };
    auto pv = [&](uint32_t half, const uint4 (&va)[4][2], const uint4 (&pt)[terms][2]) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int t = 0; t < terms; ++t)
#pragma unroll
                for (uint32_t mt = 0; mt < 4; ++mt)
                    o[4 * half + mt] = mfma<F16>(va[mt][h], pt[t][h], o[4 * half + mt]);
    };
    // causal mask and maxima of block kb's scores, which become sp
    auto stats = [&](uint32_t kb, const f32x16_t& s) {
        sp = s;
        const uint32_t key0 = kb * block_keys;
        if (key0 + block_keys - 1 > pos_lo) {
            asm volatile(""); // a branch: most blocks end before the diagonal
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const uint32_t kpos = key0 + 16 * (r >> 3) + 8 * g + (r & 7);
                if (kpos > qpos)
                    sp[r] = -__builtin_inff();
            }
        }
        mx = lane_max(sp);
        return __any(mx > m_limit);
    };
    auto rescale = [&]() {
        const float m_new = fmaxf(m, pair_max(mx));
        const float alpha = m_new == -__builtin_inff()
            ? 1.0f
            : __builtin_amdgcn_exp2f((m - m_new) * c); // 0 at the start
        l *= alpha;
        m = m_new;
        m_limit = m_new + rescale_raw;
#pragma unroll
        for (uint32_t mt = 0; mt < tiles_o; ++mt) {
            o[mt] *= alpha;
            asm volatile("" : "+a"(o[mt])); // one accumulator at a time, see pin
        }
    };

    // Before the loop: blocks b .. b + 3 of K and b .. b + 2 of V, those that
    // the first two iterations read first.
    uint32_t pk0, pk1, pw0, pw1; // pages of the block whose K, and V, is loaded next
    {
        const uint32_t b = kb_begin;
        uint32_t pg[4][2];
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) {
            pg[i][0] = page_of(2 * (b + i));
            pg[i][1] = page_of(2 * (b + i) + 1);
        }
        auto first_k = [&](uint32_t i) {
            if (b + i < kb_end)
                load_k(b + i, pg[i][0], pg[i][1]);
        };
        auto first_v = [&](uint32_t i) {
            if (b + i < kb_end)
                load_v(b + i, pg[i][0], pg[i][1]);
        };
        first_k(0);
        first_k(1);
        first_v(0);
        first_k(2);
        first_v(1);
        first_k(3);
        first_v(2);
        if (b + 3 < kb_end)
            __builtin_amdgcn_s_waitcnt(0x4F74); // vmcnt(20): K(b) and K(b + 1) have landed
        else
            wait_all_but(0);
        __syncthreads();
        read_k(b);
        const f32x16_t s = qk();
        read_k(min(b + 1, kb_end - 1));
        stats(b, s);
        rescale();
        pk0 = page_of(2 * (b + 4));
        pk1 = page_of(2 * (b + 4) + 1);
        pw0 = pg[3][0];
        pw1 = pg[3][1];
        wait_all_but(b + 3 < kb_end ? 3 * regions : 0); // K(b + 2) and V(b)
        __syncthreads();
    }
    // K(kb + 3) takes the stage of K(kb - 1), last read (into registers) in
    // iteration kb - 2, and V(kb + 2) that of V(kb - 2), last read in iteration
    // kb - 1; a barrier lies between in both cases. The wait leaves in flight
    // what the wave issued after K(kb + 2): V(kb + 1), K(kb + 3) and V(kb + 2).
    // Q^T and O^T stay in the accumulation registers (matrix operands may; the
    // 256 others hold K, V, scores and probabilities): left to itself the
    // compiler keeps O^T in the others and spills Q^T.
    auto pin = [&]() {
#pragma unroll
        for (uint32_t ks = 0; ks < k_steps; ++ks)
            asm volatile("" : "+a"(qr[ks]));
#pragma unroll
        for (uint32_t mt = 0; mt < tiles_o; ++mt)
            asm volatile("" : "+a"(o[mt]));
    };
    for (uint32_t kb = kb_begin + 1; kb < kb_end; ++kb) {
        pin();
        const bool more_k = kb + 3 < kb_end, more_v = kb + 2 < kb_end;
        const uint32_t newest = (more_v ? 2 * regions : 0) + (more_k ? regions : 0);
        if (more_k)
            load_k(kb + 3, pk0, pk1);
        if (more_v)
            load_v(kb + 2, pw0, pw1);
        uint4 va[4][2], vb[4][2], pt[terms][2];
        read_v(kb - 1, 0, va);
        const f32x16_t s = qk(); // matrix: block kb
        probabilities(pt);       // vector: block kb - 1
        read_v(kb - 1, 1, vb);
        pv(0, va, pt); // matrix: block kb - 1
        read_k(min(kb + 1, kb_end - 1)); // past the range's end: any staged block
        pv(1, vb, pt);
        pw0 = pk0;
        pw1 = pk1;
        pk0 = page_of(2 * (kb + 4));
        pk1 = page_of(2 * (kb + 4) + 1);
        const bool grew = stats(kb, s); // vector: block kb
        wait_all_but(newest);
        __syncthreads();
        if (grew)
            rescale();
    }
    {
        uint4 va[4][2], pt[terms][2];
        probabilities(pt);
#pragma unroll
        for (uint32_t half = 0; half < 2; ++half) {
            read_v(kb_end - 1, half, va);
            pv(half, va, pt);
        }
    }

    float lt = l + __shfl_xor(l, 32); // the query's denominator (both lane halves)
    if (n_parts > 1) {
        // The hand-over of kernels_prefill.hip, with 65 chunks of four floats per
        // (range, query vector): [max, denominator, 0, 0], then acc[4j .. 4j + 3].
        const uint32_t pair = (rest * passes + pass) * kv_heads + kvh;
        const uint32_t qv = wave * 32 + n;
        constexpr uint32_t QV = 32 * waves, chunks = dim / 4 + 1;
        const __amdgpu_buffer_rsrc_t rs = record_rsrc(
            split_scratch.records + (uint64_t)pair * n_split * (chunks * QV * 4),
            n_split * chunks * QV * 16);
        auto off = [&](uint32_t share, uint32_t chunk) {
            return ((share * chunks + chunk) * QV + qv) * 16u;
        };
#pragma unroll
        for (uint32_t mt = 0; mt < tiles_o; ++mt)
#pragma unroll
            for (uint32_t quad = 0; quad < 4; ++quad)
                agent_store4(rs, off(part, 1 + 8 * mt + 2 * quad + g), o[mt][4 * quad],
                             o[mt][4 * quad + 1], o[mt][4 * quad + 2], o[mt][4 * quad + 3]);
        if (g == 0)
            agent_store4(rs, off(part, 0), m, lt, 0.0f, 0.0f);
        wait_vector_memory();
        __syncthreads(); // also: every wave is past its LDS reads
        uint32_t* const last_flag = reinterpret_cast<uint32_t*>(lds);
        if (tid == 0) {
            const uint32_t before = __hip_atomic_fetch_add(split_scratch.arrivals + pair, 1u,
                                                           __ATOMIC_RELAXED,
                                                           __HIP_MEMORY_SCOPE_AGENT);
            const uint32_t last = before == n_parts - 1;
            if (last)
                __hip_atomic_store(split_scratch.arrivals + pair, 0u, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
            *last_flag = last;
        }
        __syncthreads();
        if (!*last_flag)
            return;
        float M = -__builtin_inff();
        auto weight = [&](float ms, float to) { // 0 for a range that attended nothing
            return ms == -__builtin_inff() ? 0.0f : __builtin_amdgcn_exp2f((ms - to) * c);
        };
        lt = 0.0f;
#pragma unroll
        for (uint32_t mt = 0; mt < tiles_o; ++mt)
            o[mt] = f32x16_t {};
        for (uint32_t s = 0; s < n_parts; ++s) {
            const u32x4_t hd = agent_load4(rs, off(s, 0));
            const float ms = __uint_as_float(hd[0]);
            const float m_new = fmaxf(M, ms);
            const float keep = weight(M, m_new), w = weight(ms, m_new);
            M = m_new;
            lt = lt * keep + __uint_as_float(hd[1]) * w;
            // a quarter of the range's record at a time (64 registers)
#pragma unroll
            for (uint32_t mt = 0; mt < tiles_o; mt += 2) {
                u32x4_t v[8];
#pragma unroll
                for (uint32_t j = 0; j < 8; ++j)
                    v[j] = agent_load4(rs, off(s, 1 + 8 * mt + 2 * j + g));
#pragma unroll
                for (uint32_t j = 0; j < 8; ++j)
#pragma unroll
                    for (uint32_t e = 0; e < 4; ++e) {
                        const uint32_t r = 4 * (j % 4) + e;
                        o[mt + j / 4][r] = o[mt + j / 4][r] * keep + __uint_as_float(v[j][e]) * w;
                    }
            }
        }
    }

    const float inv = 1.0f / lt;
    // 0 unless some result of the query is infinite or NaN (either lane half)
    float odd = inv * 0.0f;
#pragma unroll
    for (uint32_t mt = 0; mt < tiles_o; ++mt)
#pragma unroll
        for (int r = 0; r < 16; ++r)
            odd = __builtin_fmaf(o[mt][r], 0.0f, odd);
    const uint64_t odd_lanes = __ballot(valid && odd != 0.0f);
    const uint32_t alone = (uint32_t)odd_lanes | (uint32_t)(odd_lanes >> 32);
    uint16_t* dst = out + qoff;
    if (valid && !(alone >> n & 1)) {
#pragma unroll
        for (uint32_t mt = 0; mt < tiles_o; ++mt)
#pragma unroll
            for (uint32_t quad = 0; quad < 4; ++quad) {
                const uint32_t f = 32 * mt + 8 * quad + 4 * g;
                float x[4] = { o[mt][4 * quad] * inv, o[mt][4 * quad + 1] * inv,
                               o[mt][4 * quad + 2] * inv, o[mt][4 * quad + 3] * inv };
                if (gate) { // sigmoid_mul (src/qwen/qwen_layer.cc:204) in the epilogue
                    const uint2 gv = *reinterpret_cast<const uint2*>(gate + qoff + f);
                    const uint32_t w[2] = { gv.x, gv.y };
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        x[e] *= sigmoid(half_value<F16>((uint16_t)(w[e / 2] >> (16 * (e % 2)))));
                }
                *reinterpret_cast<uint2*>(dst + f) =
                    make_uint2(pack2<F16>(x[0], x[1]), pack2<F16>(x[2], x[3]));
            }
    }
    // (the loop out of the way: 62.4 us in all with two-term probabilities, 63.3 in line)
    if (__builtin_expect(alone == 0, 1))
        return;
    const size_t first = (size_t)(row0 + rb * 32) * q_stride + (size_t)head * dim;
    for (uint32_t left = alone; left;) {
        uint32_t some = left; // the lowest alone_queries of them
#pragma unroll
        for (uint32_t i = 0; i < alone_queries; ++i)
            left &= left - 1;
        some ^= left;
        attend_alone<F16>(static_cast<const uint16_t*>(p.keys) + base_elems,
                          static_cast<const uint16_t*>(p.values) + base_elems, table, F, some,
                          pos_lo, q + first, q_stride, c, gate ? gate + first : nullptr,
                          out + first, lane);
    }
}

template <int G>
hipError_t launch_g(hipStream_t s, const pool_view& p, const meta_view& m, uint32_t layer,
                    const void* q, uint32_t q_heads, float c, void* out, const void* gate,
                    uint32_t grid, prefill_split split)
{
    const bool far = p.layer_elems * 2 > 0xFFFFFFFFull;
    const bool f16 = p.dtype == CKV_F16;
    const auto* qq = static_cast<const uint16_t*>(q);
    auto* oo = static_cast<uint16_t*>(out);
    const auto* gg = static_cast<const uint16_t*>(gate);
    const dim3 blocks(grid), threads(64 * waves);
    if (f16 && far)
        prefill_wide_kernel<G, true, true><<<blocks, threads, 0, s>>>(p, m, layer, qq, oo, q_heads, c, gg, split);
    else if (f16)
        prefill_wide_kernel<G, true, false><<<blocks, threads, 0, s>>>(p, m, layer, qq, oo, q_heads, c, gg, split);
    else if (far)
        prefill_wide_kernel<G, false, true><<<blocks, threads, 0, s>>>(p, m, layer, qq, oo, q_heads, c, gg, split);
    else
        prefill_wide_kernel<G, false, false><<<blocks, threads, 0, s>>>(p, m, layer, qq, oo, q_heads, c, gg, split);
    return hipGetLastError();
}

// Query heads a workgroup covers of a GQA group.
uint32_t wide_heads(uint32_t group)
{
    return std::min(group, 4u);
}

} // namespace

// One workgroup per compute unit: if the tiles do not fill them, each tile's
// keys are split between as many workgroups as do (at most split_max).
// CKV_PREFILL_SPLIT overrides.
prefill_shape_info prefill_wide_plan(const pool_view& p, const meta_view& m, uint32_t q_heads,
                                     int cu_count, uint32_t min_blocks)
{
    prefill_shape_info plan { waves, 1, min_blocks, 0, 0 };
    const uint32_t group = q_heads / p.kv_heads, G = wide_heads(group);
    // row_blocks[i]: the tiles' workgroups of 32 << i rows
    const uint64_t busy = (uint64_t)m.row_blocks[G == 4 ? 0 : G == 2 ? 1 : 2] * (group / G) * p.kv_heads;
    uint64_t split = busy && cu_count > 0 ? (uint64_t)cu_count / busy : 1;
    if (const char* forced = std::getenv("CKV_PREFILL_SPLIT"))
        split = (uint64_t)std::max(1L, std::strtol(forced, nullptr, 10));
    // records are kept for every workgroup of the grid, those past a short
    // tile's rows included: within 128 MiB
    const uint64_t grid = (uint64_t)m.n_tiles * (prefill_tile_rows * G / (32 * waves)) * (group / G)
        * p.kv_heads;
    const uint64_t floats = grid * (32 * waves) * (dim + 4);
    const uint64_t room = std::max<uint64_t>(1, ((uint64_t)128 << 20) / sizeof(float) / std::max<uint64_t>(floats, 1));
    plan.n_split = (uint32_t)std::clamp<uint64_t>(std::min(split, room), 1, split_max);
    if (plan.n_split > 1) {
        plan.records_floats = floats * plan.n_split;
        plan.counters = grid;
    }
    return plan;
}

hipError_t launch_prefill_wide(hipStream_t s, const pool_view& p, const meta_view& m,
                               uint32_t layer, const void* q, uint32_t q_heads, float scale,
                               void* out, const void* gate, prefill_split split)
{
    const uint32_t group = q_heads / p.kv_heads, G = wide_heads(group);
    const uint64_t grid = (uint64_t)m.n_tiles * (prefill_tile_rows * G / (32 * waves)) * (group / G)
        * p.kv_heads * split.n_split;
    if (!grid)
        return hipSuccess;
    if (grid > 0x7FFFFFFFull)
        return hipErrorInvalidValue;
    const float c = scale * log2e;
    switch (G) {
    case 1:
        return launch_g<1>(s, p, m, layer, q, q_heads, c, out, gate, (uint32_t)grid, split);
    case 2:
        return launch_g<2>(s, p, m, layer, q, q_heads, c, out, gate, (uint32_t)grid, split);
    default:
        return launch_g<4>(s, p, m, layer, q, q_heads, c, out, gate, (uint32_t)grid, split);
    }
}

} // namespace ckv

// Measurement-to-detection-event kernels for gfx950 (MI355X).
//
// m2d_kernel converts tiles of 32 shots: 32-column blocks of the measurement rows are loaded one per lane, turned
// into measurement-major words in LDS (word m = measurement m of the tile's 32 shots) by a transpose in
// registers; each output column is the XOR of its measurements' words, inverted when its reference parity is 1
// (semantics in m2d.h), and the column words are transposed back, again one block per lane, and stored. HBM
// traffic is the minimum: each shot's measurement row is read once and its output rows written once.
//
// Also here: the windowed conversion kernel (a ring of recent measurement words per tile, for records
// longer than LDS holds; m2d.h) and the measurement sampler's expansion kernel (detection events to
// measurement records; expand.h).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "bitops.h"
#include "launch_util.h"
#include "m2d.h"

using namespace sa;

namespace {

constexpr int M2D_NT = 512;   // whole-record conversion and expansion: lanes per workgroup

// Copies staged rows [0, valid) (pitch P bytes in LDS) to bytes [off, off + nbytes) of shot rows s0 + r
// as 4-byte stores at any byte alignment (the HSA runtime enables unaligned global access; the
// compiler emits global_store_dword for an align-1 word): lane w of a wave takes bytes [4w, 4w + 4),
// so one store instruction writes 256 contiguous bytes of a row; the wave's rows step by NTHREADS /
// 64. A tail of 1 to 3 bytes at the end of a row is written byte by byte.
typedef uint32_t unaligned_u32 __attribute__((aligned(1)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
template <uint32_t NTHREADS, uint32_t P>
__device__ __forceinline__ void flush_words(const uint8_t *img, uint8_t *dst, uint64_t stride, uint32_t off,
                                            uint32_t nbytes, uint64_t s0, uint32_t valid) {
    constexpr uint32_t RG = NTHREADS / 64;
    static_assert(P % 4 == 0 && NTHREADS % 64 == 0, "word-aligned staging rows, whole waves");
    const uint32_t b = 4 * (threadIdx.x % 64), r0 = threadIdx.x / 64;
    if (b >= nbytes) return;
    uint8_t *const base = dst + s0 * stride + off + b;
    const uint8_t *const src = img + b;
    if (b + 4 <= nbytes) {
        for (uint32_t r = r0; r < valid; r += RG) {
            const uint32_t x = *reinterpret_cast<const uint32_t *>(src + r * P);
            __builtin_nontemporal_store(x, reinterpret_cast<unaligned_u32 *>(base + r * stride));
        }
    } else {
        for (uint32_t r = r0; r < valid; r += RG) {
            for (uint32_t k = 0; b + k < nbytes; k++) __builtin_nontemporal_store(src[r * P + k], base + r * stride + k);
        }
    }
}

// Row words of one lane: x[s] = bytes [4b, 4b + 4) of row s of a subtile (row_bytes - 4 .. row_bytes, shifted
// down, where the row ends first and `exact` forbids reading past it), for the subtile's rows up to `valid`;
// later rows repeat the last valid one (their bits belong to shots that are never written). Row s is at
// base + s * stride + off with `base` and `stride` the same for the whole workgroup, so a row costs a scalar
// add. Any alignment (the HSA runtime runs with unaligned global access on); a wave's lanes read consecutive
// words of a row.
__device__ __forceinline__ void load_rows(uint32_t (&x)[32], const uint8_t *base, uint64_t stride, uint32_t off,
                                          uint32_t row_bytes, uint32_t b, bool exact, uint32_t valid) {
    if (exact && row_bytes < 4) {
#pragma unroll
        for (uint32_t s = 0; s < 32; s++) {
            const uint8_t *r = base + (s < valid ? s : valid - 1) * stride + off;
            uint32_t v = 0;
            for (uint32_t k = 0; k < row_bytes; k++) v |= (uint32_t)r[k] << (8 * k);
            x[s] = v;
        }
        return;
    }
    const uint32_t at = exact && 4 * b + 4 > row_bytes ? row_bytes - 4 : 4 * b;
    if (valid == 32) {
#pragma unroll
        for (uint32_t s = 0; s < 32; s++)
            x[s] = *reinterpret_cast<const unaligned_u32 *>(base + s * stride + (off + at));
    } else {
#pragma unroll
        for (uint32_t s = 0; s < 32; s++)
            x[s] = *reinterpret_cast<const unaligned_u32 *>(base + (s < valid ? s : valid - 1) * stride + (off + at));
    }
    if (exact) {
        const uint32_t sh = 8 * (4 * b - at);
#pragma unroll
        for (uint32_t s = 0; s < 32; s++) x[s] >>= sh;
    }
}

// Stores a lane's words of a subtile's rows: bytes [4b, 4b + 4) of the row_bytes bytes of row s from x[s];
// addresses as in load_rows. A row's last word of 1 to 3 bytes goes out as the row's last four bytes, the missing
// ones from the lane before (which holds the word before and writes the same bytes), or byte by byte where that
// lane belongs to another wave.
__device__ __forceinline__ void store_rows(uint32_t (&x)[32], uint8_t *base, uint64_t stride, uint32_t off,
                                           uint32_t b, uint32_t row_bytes, uint32_t valid) {
    const uint32_t left = row_bytes - 4 * b;
    uint32_t at = off + 4 * b;
    bool single = false;
    if (__any(left < 4)) {
        single = left < 4 && (b == 0 || (threadIdx.x & 63) == 0);
        const bool join = left < 4 && !single;
#pragma unroll
        for (uint32_t s = 0; s < 32; s++) {
            const uint32_t before = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x[s], 0x138, 0xF, 0xF, false);
            const uint32_t last = __builtin_amdgcn_alignbyte(x[s], before, left & 3u);
            x[s] = join ? last : x[s];
        }
        if (join) at = off + row_bytes - 4;
    }
    if (!single) {
        if (valid == 32) {
#pragma unroll
            for (uint32_t s = 0; s < 32; s++) *reinterpret_cast<unaligned_u32 *>(base + s * stride + at) = x[s];
        } else {
#pragma unroll
            for (uint32_t s = 0; s < 32; s++)
                if (s < valid) *reinterpret_cast<unaligned_u32 *>(base + s * stride + at) = x[s];
        }
    } else {
#pragma unroll
        for (uint32_t s = 0; s < 32; s++) {
            if (s >= valid) continue;
            uint8_t *const p = base + s * stride + at;
            p[0] = (uint8_t)x[s];
            if (left > 1) p[1] = (uint8_t)(x[s] >> 8);
            if (left > 2) p[2] = (uint8_t)(x[s] >> 16);
        }
    }
}

// Rows on lanes: a half-wave's lane loads, or stores, the word of its own row (row < valid) of one block. For launches so
// small that a lane per block leaves most of the chip idle (convert_lanes_by_rows, expand_lanes_by_rows).
__device__ __forceinline__ uint32_t load_row(const uint8_t *r, uint32_t row_bytes, uint32_t b, bool exact) {
    if (exact && row_bytes < 4) {
        uint32_t v = 0;
        for (uint32_t k = 0; k < row_bytes; k++) v |= (uint32_t)r[k] << (8 * k);
        return v;
    }
    const uint32_t at = exact && 4 * b + 4 > row_bytes ? row_bytes - 4 : 4 * b;
    return *reinterpret_cast<const unaligned_u32 *>(r + at) >> (8 * (4 * b - at));
}
__device__ __forceinline__ void store_row(uint32_t v, uint8_t *r, uint32_t row_bytes, uint32_t b) {
    const uint32_t left = row_bytes - 4 * b;
    r += 4 * b;
    if (left >= 4) {
        *reinterpret_cast<unaligned_u32 *>(r) = v;
    } else {
        r[0] = (uint8_t)v;
        if (left > 1) r[1] = (uint8_t)(v >> 8);
        if (left > 2) r[2] = (uint8_t)(v >> 16);
    }
}
// Four consecutive blocks of a lane's row at once, from block b on (those past `blocks` are not used): a half-wave's 32
// loads, or stores, each touch a line of their own whatever their width.
typedef uint32_t __attribute__((ext_vector_type(4), aligned(1))) unaligned_u32x4;
__device__ __forceinline__ void load_row4(uint32_t (&x)[4], const uint8_t *r, uint32_t row_bytes, uint32_t b, uint32_t blocks,
                                          bool exact) {
    if (!exact || 4 * b + 16 <= row_bytes) {
        const u32x4 v = *reinterpret_cast<const unaligned_u32x4 *>(r + 4 * b);
#pragma unroll
        for (uint32_t k = 0; k < 4; k++) x[k] = v[k];
    } else {
#pragma unroll
        for (uint32_t k = 0; k < 4; k++) x[k] = b + k < blocks ? load_row(r, row_bytes, b + k, exact) : 0u;
    }
}
// Loads row blocks [0, blocks) of each subtile into its words from word `at` on: a block a half-wave where all fit at once,
// else four.
template <int NT>
__device__ __forceinline__ void load_by_rows(uint32_t *words, uint32_t subw, uint32_t at, const uint8_t *in,
                                             uint64_t stride, uint32_t row_bytes, uint32_t blocks, bool exact,
                                             uint32_t shots) {
    const uint32_t lane = threadIdx.x & 31, subs = (shots + 31) / 32;
    if (subs * blocks <= NT / 32) {
        const uint32_t i = threadIdx.x >> 5;
        if (i < subs * blocks) {
            const uint32_t t = i / blocks, b = i - t * blocks;
            const uint32_t x = load_row(in + min(32 * t + lane, shots - 1) * stride, row_bytes, b, exact);
            words[t * subw + at + 33 * b + lane] = transpose32(x, lane);
        }
        return;
    }
    const uint32_t groups = (blocks + 3) / 4;
    for (uint32_t i = threadIdx.x >> 5; i < subs * groups; i += NT / 32) {
        const uint32_t t = i / groups, b = 4 * (i - t * groups);
        uint32_t x[4];
        load_row4(x, in + min(32 * t + lane, shots - 1) * stride, row_bytes, b, blocks, exact);
#pragma unroll
        for (uint32_t k = 0; k < 4; k++) {
            const uint32_t v = transpose32(x[k], lane);
            if (b + k < blocks) words[t * subw + at + 33 * (b + k) + lane] = v;
        }
    }
}

// XOR of a column's words (first and second plane entries a, b; column `col` when listed).
// (a word's LDS address, base + 4 * index, is one multiply-add of a 16-bit half of the entry).
__device__ __forceinline__ uint32_t terms_word(const uint32_t *w, uint32_t a) {
    typedef __attribute__((address_space(3))) const uint32_t lds_cu32;
    const uint32_t base = (uint32_t)(uintptr_t)(lds_cu32 *)w;
    uint32_t lo, hi;
    asm("v_mad_u32_u16 %0, %1, 4, %2" : "=v"(lo) : "v"(a), "v"(base));
    asm("v_mad_u32_u16 %0, %1, 4, %2 op_sel:[1,0,0,0]" : "=v"(hi) : "v"(a), "v"(base));
    return *(lds_cu32 *)(uintptr_t)lo ^ *(lds_cu32 *)(uintptr_t)hi;
}
__device__ __forceinline__ uint32_t listed_word(const M2dParams &P, const uint32_t *w, uint32_t col) {
    const uint2 rec = P.cols[col];
    const uint32_t n = rec.x & M2D_INDEX_MASK;
    const uint4 *q = reinterpret_cast<const uint4 *>(P.ovf + rec.y);
    uint32_t v = 0;
    for (uint32_t u = 0; u < n; u += 4) {
        const uint4 a = q[u / 4];
        v ^= w[m2d_padded(a.x)] ^ w[m2d_padded(a.y)] ^ w[m2d_padded(a.z)] ^ w[m2d_padded(a.w)];
    }
    return v;
}

// Rows on lanes: each half-wave makes B consecutive blocks of 32 output columns of a subtile (a lane a column, its entry
// from the table by columns), transposes them and stores each row's words. The first blocks' entries are loaded
// before the workgroup's rows are.
template <uint32_t B>
struct ColumnEntries {
    uint2 e[B];
    uint32_t invert[B];
    __device__ __forceinline__ void load(const M2dParams &P, uint32_t nb, uint32_t b) {
#pragma unroll
        for (uint32_t k = 0; k < B; k++) {
            const uint32_t c = min(b + k, nb - 1);
            e[k] = P.entries[32 * c + (threadIdx.x & 31)];
            invert[k] = P.block_info[c].x;
        }
    }
};
template <bool SLOW, int NT, uint32_t B>
__device__ __forceinline__ void store_by_rows(const M2dParams &P, const uint32_t *words, uint32_t subw, uint64_t s0,
                                              uint32_t shots, ColumnEntries<B> &c) {
    const uint32_t lane = threadIdx.x & 31, subs = (shots + 31) / 32;
    const uint32_t nb = (P.n_out + 31) / 32, groups = (nb + B - 1) / B, row_bytes = (P.n_out + 7) / 8;
    for (uint32_t i = threadIdx.x >> 5; i < subs * groups; i += NT / 32) {
        const uint32_t t = i / groups, b = B * (i - t * groups);
        const uint32_t *const w = words + t * subw;
        if (i >= NT / 32) c.load(P, nb, b);
        uint32_t x[B];
#pragma unroll
        for (uint32_t k = 0; k < B; k++) {
            if (SLOW && c.e[k].x == 0xFFFFFFFFu) x[k] = b + k < nb ? listed_word(P, w, 32 * (b + k) + lane) : 0u;
            else x[k] = terms_word(w, c.e[k].x) ^ terms_word(w, c.e[k].y);
        }
#pragma unroll
        for (uint32_t k = 0; k < B; k++) {
            x[k] = transpose32(x[k], lane) ^ c.invert[k];
            const uint32_t live = P.n_out - min(32 * (b + k), P.n_out);
            if (live < 32) x[k] &= (1u << live) - 1;
        }
        if (32 * t + lane >= shots) continue;
        uint8_t *const r = P.out + (s0 + 32 * t + lane) * P.out_stride;
        if (B == 4 && 4 * b + 16 <= row_bytes) {
            const u32x4 v = {x[0], x[B > 1 ? 1 : 0], x[B > 2 ? 2 : 0], x[B > 3 ? 3 : 0]};
            *reinterpret_cast<unaligned_u32x4 *>(r + 4 * b) = v;
        } else {
#pragma unroll
            for (uint32_t k = 0; k < B; k++)
                if (b + k < nb) store_row(x[k], r, row_bytes, b + k);
        }
    }
}

// Separate observable rows (a few columns) of a workgroup's shots: one lane per shot and byte.
template <bool SLOW, int NT>
__device__ __forceinline__ void store_observables(const M2dParams &P, const uint32_t *words, uint32_t subw, uint64_t s0,
                                                  uint32_t shots) {
    const uint32_t obytes = (P.n_obs + 7) / 8;
    for (uint32_t i = threadIdx.x; i < shots * obytes; i += NT) {
        const uint32_t shot = i / obytes, j = i - shot * obytes;
        const uint32_t *const w = words + (shot / 32) * subw;
        uint32_t v = 0;
        for (uint32_t k = 0; k < 8 && 8 * j + k < P.n_obs; k++) {
            const uint32_t col = P.num_det + 8 * j + k, b = col / 32, r = col % 32;
            const uint2 info = P.block_info[b];
            const uint32_t a = P.terms[(size_t)r * P.total_blocks + b];
            uint32_t x;
            if (SLOW && a == 0xFFFFFFFFu) x = listed_word(P, w, col);
            else x = terms_word(w, a) ^ (info.y ? terms_word(w, P.terms[(size_t)(32 + r) * P.total_blocks + b]) : 0u);
            v |= (((x >> (shot % 32)) ^ (info.x >> r)) & 1u) << k;
        }
        P.obs[(s0 + shot) * P.obs_stride + j] = (uint8_t)v;
    }
}

// Whole-record conversion. A workgroup takes P.group subtiles of 32 shots; its work items are 32-column blocks of
// a subtile, one lane each. A lane loads its block's word of all 32 rows (32 loads in flight, a wave's lanes on
// consecutive words of the same row), transposes them in registers and puts the 32 measurement words into LDS;
// after a barrier it XORs 32 output columns together from LDS, transposes those and stores each row's word, a
// wave again on consecutive words of a row. Nothing is staged and, but for the columns of more than four terms
// (summed into slots between two more barriers), one barrier per workgroup is all.
// What bounds it: HBM and, for output rows of odd width, their stores (1,951-byte rows written 4 bytes a lane
// take 0.47 ms per 2^20 where 1,948-byte rows take 0.34; with non-temporal stores 0.77). Blocks on lanes
// rather than rows on lanes (32x32 transposes across half-waves, output staged in LDS 64 blocks at a time) take
// 0.96 instead of 1.53 ms per 2^20 shots at d=25 (4.3 TB/s); without its loads and stores the kernel takes 0.52.
// Resident workgroups that prefetch the next tile's rows spill and wait for their stores: 2.1 ms.
template <bool SLOW, int ROWS_NT>
__global__ __launch_bounds__(ROWS_NT ? ROWS_NT : M2D_NT, 4) void m2d_kernel(M2dParams P) {
    constexpr bool ROWS = ROWS_NT > 0;
    constexpr int NT = ROWS ? ROWS_NT : M2D_NT;
    extern __shared__ __align__(16) uint32_t words[];
    const uint32_t tid = threadIdx.x, G = P.group;
    const uint64_t s0 = (uint64_t)xcd_tile(blockIdx.x, gridDim.x) * 32 * G;
    const uint64_t left = P.shots - s0;
    const uint32_t shots = left < 32 * G ? (uint32_t)left : 32 * G;
    const uint32_t subs = (shots + 31) / 32;
    const uint32_t subw = m2d_subtile_words(P.blocks, P.sweep_blocks, P.spill_slots);
    const uint32_t zero = m2d_padded(m2d_zero_word(P.blocks, P.sweep_blocks));
    for (uint32_t i = tid; i < subs; i += NT) words[i * subw + zero] = 0;
    for (uint32_t i = tid; i < subs * P.spill_slots; i += NT) {
        const uint32_t t = i / P.spill_slots;
        words[t * subw + m2d_padded(m2d_zero_word(P.blocks, P.sweep_blocks) + 4 + (i - t * P.spill_slots))] = 0;
    }

    // Rows on lanes: this half-wave's first entries, of four blocks where one a half-wave does not do.
    const uint32_t nb = (P.n_out + 31) / 32;
    const bool wide = subs * nb > NT / 32;
    ColumnEntries<4> four;
    ColumnEntries<1> one;
    if (ROWS && nb) {
        const uint32_t i = tid >> 5, groups = (nb + 3) / 4;
        if (wide) four.load(P, nb, 4 * (i % groups));
        else one.load(P, nb, i % nb);
    }

    // Rows whose stride covers whole words are read past their last byte (never past the buffer's
    // shots * stride bytes); the bits there belong to no measurement.
    if (ROWS) load_by_rows<NT>(words, subw, 0, P.in + s0 * P.in_stride, P.in_stride, P.in_row_bytes, P.blocks, !P.in_vec, shots);
    for (uint32_t i = tid; !ROWS && i < subs * P.blocks; i += NT) {
        const uint32_t t = i / P.blocks, b = i - t * P.blocks;
        uint32_t x[32];
        load_rows(x, P.in + s0 * P.in_stride, P.in_stride, 32 * t * (uint32_t)P.in_stride, P.in_row_bytes, b, !P.in_vec,
                  min(shots - 32 * t, 32u));
        transpose_rows(x);
        uint32_t *const w = words + t * subw + 33 * b;
#pragma unroll
        for (uint32_t k = 0; k < 32; k++) w[k] = x[k];
    }
    if (P.sweep_blocks) {
        const uint32_t sw0 = m2d_padded(m2d_sweep_word(P.blocks));
        const bool by_rows = ROWS && P.sweep;
        if (by_rows)
            load_by_rows<NT>(words, subw, sw0, P.sweep + s0 * P.sweep_stride, P.sweep_stride, P.sweep_row_bytes,
                         P.sweep_blocks, true, shots);
        for (uint32_t i = tid; !by_rows && i < subs * P.sweep_blocks; i += NT) {
            const uint32_t t = i / P.sweep_blocks, b = i - t * P.sweep_blocks;
            uint32_t x[32];
#pragma unroll
            for (uint32_t s = 0; s < 32; s++) x[s] = 0;
            // Without sweep data every sweep bit is 0.
            if (P.sweep)
                load_rows(x, P.sweep + s0 * P.sweep_stride, P.sweep_stride, 32 * t * (uint32_t)P.sweep_stride,
                          P.sweep_row_bytes, b, true, min(shots - 32 * t, 32u));
            transpose_rows(x);
            uint32_t *const w = words + t * subw + sw0 + 33 * b;
#pragma unroll
            for (uint32_t k = 0; k < 32; k++) w[k] = x[k];
        }
    }
    __syncthreads();
    if (P.spill_chunks) {
        for (uint32_t i = tid; i < subs * P.spill_chunks; i += NT) {
            const uint32_t t = i / P.spill_chunks;
            const uint4 c = P.spill[i - t * P.spill_chunks];
            uint32_t *const w = words + t * subw;
            atomicXor(&w[c.z], terms_word(w, c.x) ^ terms_word(w, c.y));
        }
        __syncthreads();
    }

    const uint32_t TB = P.total_blocks;
    if (ROWS) {
        if (wide) store_by_rows<SLOW, NT, 4>(P, words, subw, s0, shots, four);
        else store_by_rows<SLOW, NT, 1>(P, words, subw, s0, shots, one);
    }
    for (uint32_t i = tid; !ROWS && i < subs * nb; i += NT) {
        const uint32_t t = i / nb, b = i - t * nb;
        const uint32_t *const w = words + t * subw;
        const uint2 info = P.block_info[b];
        uint32_t x[32];
#pragma unroll
        for (uint32_t k = 0; k < 32; k++) x[k] = (P.terms + (size_t)k * TB)[b];
        if (SLOW) {
#pragma unroll
            for (uint32_t k = 0; k < 32; k++)
                x[k] = x[k] != 0xFFFFFFFFu ? terms_word(w, x[k]) : listed_word(P, w, 32 * b + k);
        } else {
#pragma unroll
            for (uint32_t k = 0; k < 32; k++) x[k] = terms_word(w, x[k]);
        }
        if (info.y) {
            // Some column of the block has a third or fourth term.
#pragma unroll
            for (uint32_t k = 0; k < 32; k++) x[k] ^= terms_word(w, (P.terms + (size_t)(32 + k) * TB)[b]);
        }
        transpose_rows(x);
        // Inverting a column flips its bit in every shot's row; columns past the last are 0.
        const uint32_t live = P.n_out - 32 * b;
        const uint32_t keep = live < 32 ? (1u << live) - 1 : 0xFFFFFFFFu;
#pragma unroll
        for (uint32_t s = 0; s < 32; s++) x[s] = (x[s] ^ info.x) & keep;
        store_rows(x, P.out + s0 * P.out_stride, P.out_stride, 32 * t * (uint32_t)P.out_stride, b, (P.n_out + 7) / 8,
                   min(shots - 32 * t, 32u));
    }
    store_observables<SLOW, NT>(P, words, subw, s0, shots);
}

// Random words of the free results: Philox4x32-10 keyed by the sampler's expansion key, counter (group of
// four free results, 64-bit tile index, stream tag).
constexpr uint32_t TAG_EXPAND = 7u << 28;

// One substitution record (layout in expand.h): words r.x .. r.w, q.x .. q.w.
__device__ __forceinline__ void expand_record(uint32_t *words, uint4 r, uint4 q) {
    uint32_t k = r.x & 0xFFFFu;
    const uint32_t n = r.x >> 16;
    if (n == 1) {
        // A chain: each later result XORs the one before it, kept in v. Its results are distinct
        // (stride w > 0) and only this record writes them, so the words it reads are the values
        // before the chain: they are read 8 at a time ahead of the writes (the last batch repeats its last
        // result), which turns the chain's dependent LDS round trips into one per 8 (24 at a time: no faster).
        uint32_t v = words[m2d_padded(k)] ^ words[m2d_padded(r.y)];
        words[m2d_padded(k)] = v;
        uint32_t j = 1;
        for (; j + 8 <= r.z; j += 8) {
            uint32_t t[8], at[8];
#pragma unroll
            for (uint32_t u = 0; u < 8; u++) {
                k += r.w;
                at[u] = m2d_padded(k);
                t[u] = words[at[u]];
            }
#pragma unroll
            for (uint32_t u = 0; u < 8; u++) {
                v ^= t[u];
                words[at[u]] = v;
            }
        }
        if (j < r.z) {
            const uint32_t last = r.z - j - 1;   // steps after this batch's first
            uint32_t t[8], at[8];
#pragma unroll
            for (uint32_t u = 0; u < 8; u++) {
                at[u] = m2d_padded(k + (min(u, last) + 1) * r.w);
                t[u] = words[at[u]];
            }
#pragma unroll
            for (uint32_t u = 0; u < 8; u++) {
                if (u <= last) v ^= t[u];
                words[at[u]] = v;
            }
        }
    } else {
        // Terms inline: all seven read together (unused ones name result 0 and are masked). XORed in with an atomic:
        // the records that a longer list was cut into add to one result in the same step.
        const uint32_t t[EXPAND_INLINE_TERMS] = {r.y, r.z, r.w, q.x, q.y, q.z, q.w};
        uint32_t v = 0, w[EXPAND_INLINE_TERMS];
#pragma unroll
        for (uint32_t u = 0; u < EXPAND_INLINE_TERMS; u++) w[u] = words[m2d_padded(t[u])];
#pragma unroll
        for (uint32_t u = 0; u < EXPAND_INLINE_TERMS; u++) v ^= u < n ? w[u] : 0u;
        atomicXor(&words[m2d_padded(k)], v);
    }
}

// Expansion of detection events into records (semantics in expand.h), laid out as m2d_kernel: E.out.group subtiles
// of 32 shots per workgroup, a lane per 32-column block of a subtile for the y rows (transposed in registers, each
// word XORed into its result's word) and again for the record rows. Between them the substitution steps run, a
// lane per record. With two workgroups per CU they are bound by latency: so the y rows and step 0's
// records load before anything else, the later steps' records are staged in LDS meanwhile (E.staged), and the
// last steps, while they have at most 64 records, run on one wave without workgroup barriers. 2^20 shots at d=25:
// 1.32 ms (3.2 TB/s of y rows read and record rows written), of which the steps are about 0.45; with rows on
// lanes, staged output and 1024-lane workgroups 1.76.
// ONE: one subtile per workgroup (no divisions by the counts).
template <bool ONE, int ROWS_NT>
__global__ __launch_bounds__(ROWS_NT ? ROWS_NT : M2D_NT, 4) void expand_kernel(ExpandDev E) {
    constexpr bool ROWS = ROWS_NT > 0;
    constexpr int NT = ROWS ? ROWS_NT : M2D_NT;
    extern __shared__ __align__(16) uint32_t words[];
    const M2dParams &P = E.out;
    const uint32_t tid = threadIdx.x, G = ONE ? 1 : P.group;
    const uint32_t block = xcd_tile(blockIdx.x, gridDim.x);
    const uint64_t s0 = (uint64_t)block * 32 * G;
    const uint64_t left = P.shots - s0;
    const uint32_t shots = left < 32 * G ? (uint32_t)left : 32 * G;
    const uint32_t subs = ONE ? 1 : (shots + 31) / 32;
    const uint32_t subw = expand_subtile_words(P.blocks);
    uint4 *const stage = reinterpret_cast<uint4 *>(words) + (G * subw + 3) / 4;
    auto split = [&](uint32_t i, uint32_t n, uint32_t &t) {
        t = ONE ? 0 : i / n;
        return i - t * n;
    };
    // y block i of the workgroup: its rows' words and its columns' slots.
    uint32_t x[32], slot[16];
    auto load_block = [&](uint32_t i) {
        uint32_t t;
        const uint32_t b = split(i, E.y_blocks, t);
        load_rows(x, E.in + s0 * E.in_stride, E.in_stride, 32 * t * (uint32_t)E.in_stride, 0, b, false,
                  min(shots - 32 * t, 32u));
#pragma unroll
        for (uint32_t k = 0; k < 16; k++) slot[k] = (E.prim + (size_t)k * E.y_blocks)[b];
    };
    if (!ROWS && tid < subs * E.y_blocks) load_block(tid);
    const uint32_t step0 = E.nsteps ? E.steps[1] : 0, staged = E.staged;
    // Step 0's records of this lane: tid and tid + NT.
    uint4 ra, qa, rb, qb;
    uint32_t sub;
    if (tid < subs * step0) {
        const uint32_t f = split(tid, step0, sub);
        ra = E.items[2 * f];
        qa = E.items[2 * f + 1];
    }
    if (tid + NT < subs * step0) {
        const uint32_t f = split(tid + NT, step0, sub);
        rb = E.items[2 * f];
        qb = E.items[2 * f + 1];
    }
    for (uint32_t i = tid; i < 2 * staged; i += NT) stage[i] = E.items[2 * step0 + i];
    for (uint32_t i = tid; i < (subs * subw + 3) / 4; i += NT) reinterpret_cast<uint4 *>(words)[i] = make_uint4(0, 0, 0, 0);
    __syncthreads();
    // Free results (distinct from every y slot, so no ordering with the y words; slots padded, in fours).
    const uint32_t k0 = (uint32_t)E.seed, k1 = (uint32_t)(E.seed >> 32), fg = (E.nfree + 3) / 4;
    for (uint32_t i = tid; i < subs * fg; i += NT) {
        uint32_t t;
        const uint32_t g = split(i, fg, t);
        const uint64_t tile = E.tile0 + (uint64_t)block * G + t;
        const uint4 at = E.free_slots[g];
        const uint4 r = philox10(make_uint4(g, (uint32_t)tile, (uint32_t)(tile >> 32), TAG_EXPAND), k0, k1);
        uint32_t *const w = words + t * subw;
        w[at.x] = r.x;
        w[at.y] = r.y;
        w[at.z] = r.z;
        w[at.w] = r.w;
    }
    // y words into their slots (two 16-bit padded indices per entry; columns past the last go to the spare word).
    const uint32_t lane = tid & 31;
    for (uint32_t i = tid >> 5; ROWS && i < subs * E.y_blocks; i += NT / 32) {
        uint32_t t;
        const uint32_t b = split(i, E.y_blocks, t), y = 32 * b + lane;
        uint32_t v = load_row(E.in + (s0 + min(32 * t + lane, shots - 1)) * E.in_stride, 0, b, false);
        v = transpose32(v, lane);
        uint32_t *const w = words + t * subw;
        atomicXor(&w[(E.prim[(size_t)(lane / 2) * E.y_blocks + b] >> (16 * (lane & 1))) & 0xFFFFu], v);
        for (uint32_t c = E.any_extra && y < E.Y ? E.extra_off[y] : 0; E.any_extra && y < E.Y && c < E.extra_off[y + 1]; c++)
            atomicXor(&w[m2d_padded(E.extra[c])], v);
    }
    for (uint32_t i = tid; !ROWS && i < subs * E.y_blocks; i += NT) {
        if (i != tid) load_block(i);
        uint32_t t;
        const uint32_t b = split(i, E.y_blocks, t);
        transpose_rows(x);
        uint32_t *const w = words + t * subw;
#pragma unroll
        for (uint32_t k = 0; k < 16; k++) {
            atomicXor(&w[slot[k] & 0xFFFFu], x[2 * k]);
            atomicXor(&w[slot[k] >> 16], x[2 * k + 1]);
        }
        if (E.any_extra) {
#pragma unroll
            for (uint32_t k = 0; k < 32; k++) {
                const uint32_t y = 32 * b + k;
                for (uint32_t c = y < E.Y ? E.extra_off[y] : 0; y < E.Y && c < E.extra_off[y + 1]; c++)
                    atomicXor(&w[m2d_padded(E.extra[c])], x[k]);
            }
        }
    }
    __syncthreads();
    // Substitution: a step's records read results of earlier steps (a chain its own, in order).
    auto step = [&](uint32_t p, uint32_t i0) {
        const uint32_t at = E.steps[p], n = E.steps[p + 1] - at;
        for (uint32_t i = i0; i < subs * n; i += NT) {
            uint32_t t;
            const uint32_t f = at + split(i, n, t);
            uint4 r, q;
            if (f - step0 < staged) {
                // An explicit LDS pointer: one that may be either becomes a flat load, which waits for both.
                typedef __attribute__((address_space(3))) const u32x4 lds_u32x4;
                lds_u32x4 *const in_lds = (lds_u32x4 *)(stage + 2 * (f - step0));
                const u32x4 a = in_lds[0], b = in_lds[1];
                r = make_uint4(a.x, a.y, a.z, a.w);
                q = make_uint4(b.x, b.y, b.z, b.w);
            } else {
                r = E.items[2 * f];
                q = E.items[2 * f + 1];
            }
            expand_record(words + t * subw, r, q);
        }
    };
    if (E.nsteps) {
        if (tid < subs * step0) {
            (void)split(tid, step0, sub);
            expand_record(words + sub * subw, ra, qa);
        }
        if (tid + NT < subs * step0) {
            (void)split(tid + NT, step0, sub);
            expand_record(words + sub * subw, rb, qb);
        }
        step(0, tid + 2 * NT);
        __syncthreads();
    }
    const uint32_t wide = ONE ? max(E.wave_step, 1u) : E.nsteps;
    for (uint32_t p = 1; p < wide; p++) {
        step(p, tid);
        __syncthreads();
    }
    if (wide < E.nsteps) {
        // The final steps on one wave: its LDS accesses complete in order.
        if (tid < 64) {
            for (uint32_t p = wide; p < E.nsteps; p++) {
                step(p, tid);
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
            }
        }
        __syncthreads();
    }
    // Records: column m is measurement word m, inverted where the reference sample is 1 (words past the last
    // measurement are zero, as are their inversion bits).
    for (uint32_t i = tid >> 5; ROWS && i < subs * P.blocks; i += NT / 32) {
        uint32_t t;
        const uint32_t b = split(i, P.blocks, t);
        const uint32_t v = transpose32(words[t * subw + 33 * b + lane], lane) ^ E.inv[b];
        if (32 * t + lane < shots) store_row(v, P.out + (s0 + 32 * t + lane) * P.out_stride, (P.n_out + 7) / 8, b);
    }
    for (uint32_t i = tid; !ROWS && i < subs * P.blocks; i += NT) {
        uint32_t t;
        const uint32_t b = split(i, P.blocks, t);
        const uint32_t *const w = words + t * subw + 33 * b;
        const uint32_t inv = E.inv[b];
#pragma unroll
        for (uint32_t k = 0; k < 32; k++) x[k] = w[k];
        transpose_rows(x);
#pragma unroll
        for (uint32_t s = 0; s < 32; s++) x[s] ^= inv;
        store_rows(x, P.out + s0 * P.out_stride, P.out_stride, 32 * t * (uint32_t)P.out_stride, b, (P.n_out + 7) / 8,
                   min(shots - 32 * t, 32u));
    }
}

// ------------------------------------------------------------------ windowed conversion
constexpr int NTW = 256;
constexpr uint32_t WIN_HALVES = NTW / 32;
constexpr uint32_t WIN_STAGE_BLOCKS = 64;                 // output blocks staged per flush (256 bytes per row)
constexpr uint32_t WIN_PITCH = WIN_STAGE_BLOCKS * 4 + 4;  // LDS bytes per staged row

// A column word from the ring: term m is ring word m & mask; overflow padding (an index >= M) is 0.
__device__ __forceinline__ uint32_t ring_column_word(const M2dParams &P, const uint32_t *ring, uint32_t mask,
                                                     uint32_t M, uint2 r) {
    const uint32_t c = (r.x >> 28) & 3u;
    uint32_t v;
    if (c == 3) {
        v = 0;
        const uint32_t n = r.x & M2D_INDEX_MASK;
        const uint4 *q = reinterpret_cast<const uint4 *>(P.ovf + r.y);
        for (uint32_t t = 0; t < n; t += 4) {
            const uint4 a = q[t / 4];
            v ^= (a.x < M ? ring[a.x & mask] : 0u) ^ (a.y < M ? ring[a.y & mask] : 0u) ^
                 (a.z < M ? ring[a.z & mask] : 0u) ^ (a.w < M ? ring[a.w & mask] : 0u);
        }
    } else {
        const uint32_t w0 = ring[(r.x & M2D_INDEX_MASK) & mask], w1 = ring[r.y & mask];
        v = (c >= 1 ? w0 : 0u) ^ (c == 2 ? w1 : 0u);
    }
    return (r.x & M2D_INVERT) ? ~v : v;
}

// Output blocks are staged a pass at a time: up to WIN_PASS blocks, block b + u * WIN_HALVES + half
// on half-wave `half` for u < WIN_UNROLL, each lane producing one column of its block.
constexpr uint32_t WIN_UNROLL = 4;
constexpr uint32_t WIN_PASS = WIN_HALVES * WIN_UNROLL;

// Column records of a pass of n blocks from block b; lanes past n or past the part's columns load the
// zero record (an address select, so the loads stay in flight until the records are used).
__device__ __forceinline__ void win_records(const M2dParams &P, uint2 (&r)[WIN_UNROLL], uint32_t ncols,
                                            uint32_t col0, uint32_t zero_rec, uint32_t b, uint32_t n) {
    const uint32_t half = threadIdx.x >> 5, lane = threadIdx.x & 31;
#pragma unroll
    for (uint32_t u = 0; u < WIN_UNROLL; u++) {
        const uint32_t i = u * WIN_HALVES + half;
        const uint32_t c = (b + i) * 32 + lane;
        r[u] = P.cols[(i < n && c < ncols) ? col0 + c : zero_rec];
    }
}

// Emission state of one part: `staged` blocks in the staging image since the last flush, `flushed`
// blocks already written to the rows.
struct WinPart {
    uint8_t *dst;
    uint64_t stride;
    uint32_t ncols, col0, flushed, staged;
};

// Blocks of the next pass from block b of [b, b1): bounded by the staging room and WIN_PASS.
__device__ __forceinline__ uint32_t win_pass_blocks(const WinPart &W, uint32_t b, uint32_t b1) {
    const uint32_t room = WIN_STAGE_BLOCKS - W.staged, left = b1 - b;
    const uint32_t n = left < room ? left : room;
    return n < WIN_PASS ? n : WIN_PASS;
}

// Emits blocks [b, b1) of a part, the first pass from the records r (loaded by the caller for the
// pass win_pass_blocks gives), and flushes the staging image whenever it fills and, with final_flush,
// at the end. Uniform across the workgroup.
__device__ __forceinline__ void win_emit(const M2dParams &P, const uint32_t *ring, uint32_t mask, uint32_t M,
                                         uint32_t zero_rec, uint8_t *img, WinPart &W, uint32_t b, uint32_t b1,
                                         uint2 (&r)[WIN_UNROLL], uint64_t s0, uint32_t valid, bool final_flush) {
    const uint32_t half = threadIdx.x >> 5, lane = threadIdx.x & 31;
    const uint32_t pitch = (W.ncols + 7) / 8;
    uint32_t *const slot = reinterpret_cast<uint32_t *>(img + lane * WIN_PITCH);
    bool first = true;
    while (b < b1 || (final_flush && W.staged)) {
        const uint32_t n = win_pass_blocks(W, b, b1);
        if (!first) win_records(P, r, W.ncols, W.col0, zero_rec, b, n);
        first = false;
        // Every lane of a half-wave takes part in the transposes; the zero record yields 0.
#pragma unroll
        for (uint32_t u = 0; u < WIN_UNROLL; u++) {
            const uint32_t i = u * WIN_HALVES + half;
            const uint32_t x = transpose32(ring_column_word(P, ring, mask, M, r[u]), lane);
            if (i < n) slot[W.staged + i] = x;
        }
        b += n;
        W.staged += n;
        if (W.staged == WIN_STAGE_BLOCKS || (final_flush && b == b1)) {
            __syncthreads();
            const uint32_t off = 4 * W.flushed;
            const uint32_t nbytes = pitch - off < 4 * W.staged ? pitch - off : 4 * W.staged;
            flush_words<NTW, WIN_PITCH>(img, W.dst, W.stride, off, nbytes, s0, valid);
            __syncthreads();
            W.flushed += W.staged;
            W.staged = 0;
        }
    }
}

// Windowed conversion of a 32-shot tile (semantics in m2d.h). Per chunk: its 16-byte groups (one per
// half-wave, loaded during the previous chunk) go into the ring; the first pass's column records are
// loaded, then the next chunk's groups (loads complete in order, so waiting for the records leaves
// the row load in flight); then the chunk's ready blocks are emitted.
__global__ __launch_bounds__(NTW) void m2d_win_kernel(M2dParams P, M2dWindow Wn) {
    extern __shared__ __align__(16) uint32_t ring[];
    const uint32_t tid = threadIdx.x, half = tid >> 5, lane = tid & 31;
    const uint64_t s0 = (uint64_t)blockIdx.x * 32;
    const uint64_t left = P.shots - s0;
    const uint32_t valid = left < 32 ? (uint32_t)left : 32u;
    const bool have = lane < valid;
    // Lanes past the tile's shots read the tile's first row; their words are never used.
    const uint4 *row = reinterpret_cast<const uint4 *>(P.in + (s0 + (have ? lane : 0)) * P.in_stride);
    const uint32_t mask = Wn.ring_words - 1, M = P.blocks * 32;
    const uint32_t ngrp = (P.blocks + 3) / 4;
    uint8_t *const img = reinterpret_cast<uint8_t *>(ring + Wn.ring_words);
    uint32_t *const chunk_end = reinterpret_cast<uint32_t *>(img + 32 * WIN_PITCH);
    for (uint32_t i = tid; i < Wn.nchunks; i += NTW) chunk_end[i] = Wn.chunk_end[i];
    const uint32_t nb0 = (P.n_out + 31) / 32;
    constexpr uint32_t GPC = M2D_WIN_CHUNK / 128;   // 16-byte groups per chunk, one per half-wave
    static_assert(GPC == WIN_HALVES, "one group per half-wave and chunk");
    // Loads past the row's last group re-read it (their words are not stored).
    uint4 v = row[half < ngrp ? half : ngrp - 1];
    WinPart W0{P.out, P.out_stride, P.n_out, 0, 0, 0};
    uint32_t next0 = 0;
    uint2 r[WIN_UNROLL];
    for (uint32_t ch = 0; ch < Wn.nchunks; ch++) {
        const uint32_t g = ch * GPC + half;
        __syncthreads();   // the previous chunk's columns are read before its ring slots are reused
        {
            const uint32_t xs[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (uint32_t k = 0; k < 4; k++) {
                const uint32_t x = transpose32(xs[k], lane);
                if (g < ngrp) ring[((4 * g + k) * 32 + lane) & mask] = x;
            }
        }
        const uint32_t b1 = chunk_end[ch];
        win_records(P, r, W0.ncols, 0, Wn.zero_rec, next0, win_pass_blocks(W0, next0, b1));
        const uint32_t gn = g + GPC;
        v = row[gn < ngrp ? gn : ngrp - 1];
        __syncthreads();
        if (b1 > next0) win_emit(P, ring, mask, M, Wn.zero_rec, img, W0, next0, b1, r, s0, valid, false);
        next0 = b1;
    }
    if (P.n_out) {
        win_records(P, r, W0.ncols, 0, Wn.zero_rec, next0, win_pass_blocks(W0, next0, nb0));
        win_emit(P, ring, mask, M, Wn.zero_rec, img, W0, next0, nb0, r, s0, valid, true);
    }
    if (P.n_obs) {
        WinPart W1{P.obs, P.obs_stride, P.n_obs, P.num_det, 0, 0};
        const uint32_t nb1 = (P.n_obs + 31) / 32;
        win_records(P, r, W1.ncols, W1.col0, Wn.zero_rec, 0, win_pass_blocks(W1, 0, nb1));
        win_emit(P, ring, mask, M, Wn.zero_rec, img, W1, 0, nb1, r, s0, valid, true);
    }
}

}  // namespace

namespace sa {

size_t m2d_win_lds_bytes(uint32_t ring_words, uint32_t nchunks) {
    return (size_t)ring_words * 4 + 32 * WIN_PITCH + ((size_t)nchunks + 3) / 4 * 16;
}

hipError_t launch_m2d_win(const M2dParams &P, const M2dWindow &Wn, hipStream_t stream) {
    const uint64_t tiles = (P.shots + 31) / 32;
    if (tiles == 0) return hipSuccess;
    const size_t lds = m2d_win_lds_bytes(Wn.ring_words, Wn.nchunks);
    static size_t reserved = 0;
    const hipError_t e = reserve_lds(reinterpret_cast<const void *>(&m2d_win_kernel), lds, reserved);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(m2d_win_kernel, dim3((uint32_t)tiles), dim3(NTW), lds, stream, P, Wn);
    return hipGetLastError();
}

// Subtiles per workgroup: as many as fill its lanes with blocks while the words of two or more workgroups fit a CU's
// LDS (80 KB each), few enough that a small call still spreads over the chip (512 workgroups: two per CU), and
// rows of a workgroup within the 32-bit offsets its lanes use.
static uint32_t subtiles(uint64_t tiles, uint32_t blocks, size_t subtile_bytes, uint64_t widest_stride) {
    uint64_t g = std::min<uint64_t>(M2D_NT / std::max(blocks, 1u), 80 * 1024 / subtile_bytes);
    g = std::min<uint64_t>(std::min<uint64_t>(g, tiles / 512), (1ull << 31) / 32 / std::max<uint64_t>(widest_stride, 1));
    return (uint32_t)std::max<uint64_t>(g, 1);
}

// Small launches put rows on lanes (0: blocks on lanes): a lane per block takes a wave through two transposes of 500
// instructions (5 us) while most SIMDs have no wave at all. Rows on lanes pay for a line per row and group of blocks.
// Expansion, a block a half-wave. Up to 256 subtiles, one workgroup per CU, of 1024 lanes: up to four blocks for each of its
// 32 half-waves that is faster; beyond, with 512 lanes, as far as its 16 half-waves have a block or two and the launch has
// less than a wave of blocks for each SIMD. Rows | blocks on lanes: 4 blocks per subtile, 4000 shots 7.9 | 15.7 us,
// 250,000 shots 15.1 (1024 lanes: 21.8) | 25.5.
static int expand_lanes_by_rows(uint64_t tiles, uint32_t blocks) {
    if (tiles <= 256) return blocks <= 112 ? 1024 : 0;
    return blocks <= 32 && tiles * blocks * ((blocks + 15) / 16) <= 48 * 1024 ? 512 : 0;
}
// Conversion, four blocks a half-wave. One subtile a CU: 1024 lanes, while those are no more than two rounds (rows | blocks on
// lanes, 4000 shots: 69 blocks 7.5 | 9.3 us, 138 blocks 7.9 | 9.2, 193 blocks 9.1 | 9.3, 313 blocks 11.9 | 11.7). Up to four a
// CU: 512 lanes (69 blocks, 11,000 shots 9.0 | 10.7, 23,000 shots 10.9 | 14.2; 136 blocks, 11,000 shots 11.3 | 11.5, 16,000
// shots 11.9 | 11.1, 20,000 shots 14.0 | 14.7). More: by the blocks in all (31 blocks, 65,000 shots 11.7 | 14.0, 131,000
// shots 18.3 | 16.7; 69 blocks, 33,000 shots 14.3 | 13.9).
static int convert_lanes_by_rows(uint64_t tiles, uint32_t blocks) {
    if (tiles <= 256) return blocks <= 176 ? 1024 : 0;
    if (tiles <= 1024) return blocks <= (tiles <= 512 ? 120 : 144) ? 512 : 0;
    return tiles * blocks <= 68 * 1024 ? 512 : 0;
}

hipError_t launch_expand(ExpandDev E, hipStream_t stream) {
    const uint64_t tiles = (E.out.shots + 31) / 32;
    if (tiles == 0) return hipSuccess;
    const size_t sub = (size_t)expand_subtile_words(E.out.blocks) * 4;
    const int rows = expand_lanes_by_rows(tiles, std::max(E.out.blocks, E.y_blocks));
    E.out.group = subtiles(tiles, std::max(E.out.blocks, E.y_blocks), sub, std::max(E.in_stride, E.out.out_stride));
    // Records after phase 0 staged in LDS where two workgroups still fit a CU.
    size_t lds = (sub * E.out.group + 15) / 16 * 16;
    const size_t later = (size_t)E.staged * 32;
    if (lds + later <= 80 * 1024) lds += later;
    else E.staged = 0;
    const uint64_t grid = (tiles + E.out.group - 1) / E.out.group;
#define STIM_AMD_LAUNCH(ONE, ROWS)                                                                               \
    {                                                                                                            \
        static size_t reserved = 0;                                                                              \
        const hipError_t e = reserve_lds(reinterpret_cast<const void *>(&expand_kernel<ONE, ROWS>), lds, reserved); \
        if (e != hipSuccess) return e;                                                                           \
        hipLaunchKernelGGL((expand_kernel<ONE, ROWS>), dim3((uint32_t)grid), dim3(ROWS ? ROWS : M2D_NT), lds, stream, E);       \
    }
    if (rows == 1024) STIM_AMD_LAUNCH(false, 1024)
    else if (rows) STIM_AMD_LAUNCH(false, 512)
    else if (E.out.group == 1) STIM_AMD_LAUNCH(true, 0)
    else STIM_AMD_LAUNCH(false, 0)
#undef STIM_AMD_LAUNCH
    return hipGetLastError();
}

// Limit on a tile's record: its words plus 8 KB.
size_t m2d_lds_bytes(uint32_t blocks, uint32_t sweep_blocks) {
    return ((size_t)m2d_zero_word(blocks, sweep_blocks) + 4) * 4 + 32 * 260;
}

hipError_t launch_m2d(M2dParams P, hipStream_t stream) {
    const uint64_t tiles = (P.shots + 31) / 32;
    if (tiles == 0) return hipSuccess;
    const uint32_t nb = std::max(P.blocks, (P.n_out + 31) / 32);
    const size_t sub = (size_t)m2d_subtile_words(P.blocks, P.sweep_blocks, P.spill_slots) * 4;
    P.group = subtiles(tiles, nb, sub, std::max(std::max(P.in_stride, P.out_stride), P.sweep_stride));
    const size_t lds = sub * P.group;
    const uint64_t grid = (tiles + P.group - 1) / P.group;
#define STIM_AMD_LAUNCH(SLOW, ROWS)                                                                              \
    {                                                                                                            \
        static size_t reserved = 0;                                                                              \
        const hipError_t e = reserve_lds(reinterpret_cast<const void *>(&m2d_kernel<SLOW, ROWS>), lds, reserved); \
        if (e != hipSuccess) return e;                                                                           \
        hipLaunchKernelGGL((m2d_kernel<SLOW, ROWS>), dim3((uint32_t)grid), dim3(ROWS ? ROWS : M2D_NT), lds, stream, P);         \
    }
    const int rows = convert_lanes_by_rows(tiles, nb);
    if (rows == 1024 && P.slow) STIM_AMD_LAUNCH(true, 1024)
    else if (rows == 1024) STIM_AMD_LAUNCH(false, 1024)
    else if (rows && P.slow) STIM_AMD_LAUNCH(true, 512)
    else if (rows) STIM_AMD_LAUNCH(false, 512)
    else if (P.slow) STIM_AMD_LAUNCH(true, 0)
    else STIM_AMD_LAUNCH(false, 0)
#undef STIM_AMD_LAUNCH
    return hipGetLastError();
}

}  // namespace sa

// Frame-simulation kernel for gfx950 (MI355X).
//
// One workgroup owns a tile of 32*T shots. Its whole Pauli frame (X and Z rows, one T-word row per
// qubit, shots along the bits), the measurement-record ring, 256 staged detector rows and the
// observable rows live in LDS for the entire circuit. The workgroup walks the device program
// (program.h) in order; each op spreads its items (targets, pairs, detectors, noise chunks) over
// the workgroup's lanes, and ops that touch a row an earlier unsynchronized op touched are separated by a
// workgroup barrier (placed by the host compiler).
//
// Reference semantics restated here:
//   frame rules            src/stim/simulators/frame_simulator.inl:172-630
//   sparse noise           RareErrorIterator (src/stim/util_bot/probability_util.h:33-71): a Bernoulli(p)
//                          process over (site, shot) positions sampled by geometric gaps; here the
//                          positions of a tile are cut into chunks, each chunk an independent
//                          Philox4x32-10 stream (Salmon et al., SC'11), which keeps the process exact
//                          because geometric gaps are memoryless.
//   detectors/observables  frame_simulator.inl:221-252 (XOR of record rows / frame rows)
//   shot-major output      src/stim/py/numpy.pybind.cc:20-63 (bit m of shot s at byte m/8, bit m%8);
//                          the transpose is done 32x32 bits at a time across lanes.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "bitops.h"
#include "launch_util.h"
#include "program.h"
#include "rng.h"

using namespace sa;

namespace {

template <int T>
struct alignas(4 * T) Wd {
    uint32_t v[T];
};

template <int T>
__device__ __forceinline__ Wd<T> wxor(Wd<T> a, const Wd<T> &b) {
#pragma unroll
    for (int k = 0; k < T; k++) a.v[k] ^= b.v[k];
    return a;
}
template <int T>
__device__ __forceinline__ Wd<T> wzero() {
    Wd<T> r;
#pragma unroll
    for (int k = 0; k < T; k++) r.v[k] = 0;
    return r;
}
template <int T>
__device__ __forceinline__ Wd<T> &row(uint32_t *base, uint32_t r) {
    return *reinterpret_cast<Wd<T> *>(base + (size_t)r * T);
}

// Stream tags keep the counter spaces of different uses apart.
constexpr uint32_t TAG_NOISE = 0u << 28;
constexpr uint32_t TAG_RAND = 1u << 28;
constexpr uint32_t TAG_INIT = 2u << 28;
constexpr uint32_t TAG_DENSE = 3u << 28;

__device__ __forceinline__ uint32_t scalar(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }

struct Rng {
    uint32_t k0, k1;
    uint32_t tile;
    __device__ uint4 draw(uint32_t a, uint32_t b, uint32_t tag_and_id) const {
        return philox10(make_uint4(a, b, tile, tag_and_id), k0, k1);
    }
};

// Geometric gap: number of failures before the next success of a Bernoulli(p) process,
// floor(log(u) / log(1 - p)) with u uniform in (0, 1]; at most 2^30, which is past the end of every chunk.
__device__ __forceinline__ uint32_t geometric_gap(uint32_t r, float inv_log2_1mp) {
    const float u = ((float)(r >> 8) + 1.0f) * (1.0f / 16777216.0f);
    return (uint32_t)fminf(__log2f(u) * inv_log2_1mp, 1073741824.0f);
}

__device__ __forceinline__ uint32_t pick_outcome(const uint32_t *otab, uint32_t woff, uint32_t nout, uint32_t r) {
    for (uint32_t i = 0; i + 1 < nout; i++) {
        if (r <= otab[woff + 2 * i]) return otab[woff + 2 * i + 1];
    }
    return otab[woff + 2 * (nout - 1) + 1];
}

// Bernoulli(p) bits for 32 shots by comparing 24-bit uniforms bit-sliced across the word.
__device__ __forceinline__ uint32_t bernoulli_word(float p, const Rng &rng, uint32_t a, uint32_t id) {
    if (p >= 1.0f) return 0xFFFFFFFFu;
    uint32_t P = (uint32_t)(p * 16777216.0f);
    uint32_t lt = 0, eq = 0xFFFFFFFFu;
    for (int blk = 0; blk < 6; blk++) {
        uint4 r = rng.draw(a, (uint32_t)blk, TAG_DENSE | id);
        uint32_t rs[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
        for (int k = 0; k < 4; k++) {
            int bit = 23 - (blk * 4 + k);
            uint32_t pb = (P >> bit) & 1u;
            if (pb) {
                lt |= eq & ~rs[k];
                eq &= rs[k];
            } else {
                eq &= ~rs[k];
            }
        }
    }
    return lt;
}

template <int T>
struct Tile {
    uint32_t *X, *Z, *REC, *STG, *OBS, *CHAIN;
};

// Applies one noise outcome to shot s of the tile. site is the site within op.
template <int T>
__device__ __forceinline__ void apply_hit(const Tile<T> &t, const DevOp &op, const uint32_t *__restrict__ tgt,
                                          uint32_t site, uint32_t s, uint32_t code) {
    const uint32_t w = s >> 5;
    const uint32_t bit = 1u << (s & 31);
    switch (op.code & 0xFF) {
        case OP_NOISE1: {
            uint32_t q = tgt[op.toff + site];
            if (code & 1) atomicXor(&t.X[q * T + w], bit);
            if (code & 2) atomicXor(&t.Z[q * T + w], bit);
            break;
        }
        case OP_NOISE2: {
            uint32_t q1 = tgt[op.toff + 2 * site], q2 = tgt[op.toff + 2 * site + 1];
            if (code & 1) atomicXor(&t.X[q1 * T + w], bit);
            if (code & 2) atomicXor(&t.Z[q1 * T + w], bit);
            if (code & 4) atomicXor(&t.X[q2 * T + w], bit);
            if (code & 8) atomicXor(&t.Z[q2 * T + w], bit);
            break;
        }
        case OP_MFLIP:
            if (code & 1) atomicXor(&t.REC[(op.base + site) * T + w], bit);
            break;
        case OP_CORR: {
            if (!(code & 1)) break;
            uint32_t old = atomicOr(&t.CHAIN[w], bit);
            if (old & bit) break;
            for (uint32_t i = 0; i < op.base; i++) {
                uint32_t term = tgt[op.toff + i];
                uint32_t q = term & TERM_QMASK;
                if (term & TERM_X) atomicXor(&t.X[q * T + w], bit);
                if (term & TERM_Z) atomicXor(&t.Z[q * T + w], bit);
            }
            break;
        }
        case OP_HERALD: {
            uint32_t q = tgt[op.toff + site];
            if (code & 4) atomicOr(&t.REC[(op.base + site) * T + w], bit);
            if (code & 1) atomicXor(&t.X[q * T + w], bit);
            if (code & 2) atomicXor(&t.Z[q * T + w], bit);
            break;
        }
        default:
            break;
    }
}

// Writes staged rows [0, n) (entries base .. base + n) of the tile to one output.
template <int T, int NT>
__device__ void flush_rows(const uint32_t *rows, uint32_t n, uint32_t base, const DevOut &out, uint64_t shot0,
                           uint64_t shots_valid) {
    const uint32_t tid = threadIdx.x;
    if (out.packed) {
        // Blocks of 32 rows x 32 shots; each half-wave transposes one block.
        const uint32_t nblk = ((n + 31) / 32) * T;
        const uint32_t half = tid >> 5, lane = tid & 31;
        for (uint32_t b = half; b < ((nblk + NT / 32 - 1) / (NT / 32)) * (NT / 32); b += NT / 32) {
            // All lanes of a half-wave take part in the shuffles; blocks past the end are masked.
            const bool live = b < nblk;
            const uint32_t rb = live ? b / T : 0, w = live ? b % T : 0;
            const uint32_t r = rb * 32 + lane;
            uint32_t x = (live && r < n) ? rows[r * T + w] : 0u;
            x = transpose32(x, lane);
            const uint64_t shot = shot0 + w * 32 + lane;
            if (live && shot < shots_valid) {
                uint8_t *p = out.ptr + shot * out.stride + (out.col0 >> 3) + ((base + rb * 32) >> 3);
                const uint32_t remaining = n - rb * 32;
                const uint32_t nbytes = remaining >= 32 ? 4 : (remaining + 7) / 8;
                store_bytes(p, x, nbytes);
            }
        }
    } else {
        const uint32_t W = 32 * T;
        for (uint32_t i = tid; i < n * W; i += NT) {
            const uint32_t s = i / n, r = i % n;
            const uint64_t shot = shot0 + s;
            if (shot < shots_valid) {
                uint32_t bitv = (rows[r * T + (s >> 5)] >> (s & 31)) & 1u;
                out.ptr[shot * out.stride + out.col0 + base + r] = (uint8_t)(bitv + out.base_char);
            }
        }
    }
}

// One position of a sparse noise op that fired, with the words that its application needs on their way from memory.
struct Hit {
    uint32_t site, shot, code, a, b;
    bool live;
};

// Sparse noise of kind CODE (NOISE1, NOISE2, MFLIP or HERALD). The tile's (site, shot) positions are cut into chunks
// spread over all lanes (at most ~4/p positions each); each chunk walks its own geometric gaps, two hits per Philox
// block (gap, outcome, gap, outcome). A hit needs its site's qubits and its outcome from memory: both loads of both hits
// of a block are started together, and the next block is drawn while they are on their way. The outcome is the number
// of thresholds below the draw; these wait in scalar registers.
template <int T, int NT, uint32_t CODE>
__device__ __forceinline__ void sparse_noise(const Tile<T> &t, const DevOp &op, const uint32_t *__restrict__ ntgt,
                                             const uint32_t *__restrict__ otab, const Rng &rng, uint32_t oi,
                                             uint32_t clog, uint64_t N) {
    constexpr uint32_t W = 32 * T;
    constexpr uint32_t OUTCOMES = noise_outcomes(CODE);
    const uint32_t *__restrict__ tab = otab + op.woff;
    const uint32_t *__restrict__ tgt = ntgt + op.toff;
    uint32_t threshold[OUTCOMES];
#pragma unroll
    for (uint32_t i = 0; i + 1 < OUTCOMES; i++) threshold[i] = tab[2 * i];
    auto fetch = [&](bool live, uint64_t pos, uint32_t r) __attribute__((always_inline)) {
        Hit h = {0, 0, 0, 0, 0, live};
        if (!live) return h;
        h.site = (uint32_t)(pos / W);
        h.shot = (uint32_t)(pos % W);
        uint32_t k = 0;
#pragma unroll
        for (uint32_t i = 0; i + 1 < OUTCOMES; i++) k += r > threshold[i];
        h.code = tab[2 * k + 1];
        if (CODE == OP_NOISE1 || CODE == OP_HERALD) h.a = tgt[h.site];
        if (CODE == OP_NOISE2) {
            h.a = tgt[2 * h.site];
            h.b = tgt[2 * h.site + 1];
        }
        return h;
    };
    auto apply = [&](Hit h) __attribute__((always_inline)) {
        if (!h.live) return;
        const uint32_t w = h.shot >> 5, bit = 1u << (h.shot & 31);
        if (CODE == OP_MFLIP || CODE == OP_HERALD) {
            uint32_t *const rec = &t.REC[(op.base + h.site) * T + w];
            if (CODE == OP_MFLIP) {
                if (h.code & 1) atomicXor(rec, bit);
            } else if (h.code & 4) {
                atomicOr(rec, bit);
            }
        }
        if (CODE != OP_MFLIP) {
            if (h.code & 1) atomicXor(&t.X[h.a * T + w], bit);
            if (h.code & 2) atomicXor(&t.Z[h.a * T + w], bit);
        }
        if (CODE == OP_NOISE2) {
            if (h.code & 4) atomicXor(&t.X[h.b * T + w], bit);
            if (h.code & 8) atomicXor(&t.Z[h.b * T + w], bit);
        }
    };
    const uint64_t nch = (N + ((uint64_t)1 << clog) - 1) >> clog;
    for (uint64_t ch = threadIdx.x; ch < nch; ch += NT) {
        const uint64_t lo = ch << clog;
        const uint32_t len = (uint32_t)(N - lo < ((uint64_t)1 << clog) ? N - lo : (uint64_t)1 << clog);
        uint32_t pos = 0, ctr = 0;
        Hit a = {0, 0, 0, 0, 0, false}, b = a;
        while (true) {
            const uint4 r = rng.draw(ctr++, (uint32_t)ch, TAG_NOISE | oi);
            const uint32_t pa = pos + geometric_gap(r.x, op.inv_log);
            const uint32_t pb = pa + 1 + geometric_gap(r.z, op.inv_log);
            const bool la = pa < len, lb = la && pb < len;
            apply(a);
            apply(b);
            a = fetch(la, lo + pa, r.y);
            b = fetch(lb, lo + pb, r.w);
            pos = pb + 1;
            if (!lb || pos >= len) break;
        }
        apply(a);
        apply(b);
    }
}

// The same for one Pauli product of a chain (OP_CORR, a single site). No barrier parts the products of a chain: sampled
// sparsely or densely, all of them run on the first wave, in order.
template <int T, int NT>
__device__ __forceinline__ void sparse_chain(const Tile<T> &t, const DevOp &op, const uint32_t *__restrict__ ntgt,
                                             const uint32_t *__restrict__ otab, const Rng &rng, uint32_t oi,
                                             uint32_t clog, uint64_t N) {
    constexpr uint32_t W = 32 * T;
    const uint64_t nch = (N + ((uint64_t)1 << clog) - 1) >> clog;
    for (uint64_t ch = threadIdx.x; ch < nch; ch += NT) {
        const uint64_t lo = ch << clog;
        const uint32_t len = (uint32_t)(N - lo < ((uint64_t)1 << clog) ? N - lo : (uint64_t)1 << clog);
        uint32_t pos = 0, ctr = 0;
        while (pos < len) {
            const uint4 r = rng.draw(ctr++, (uint32_t)ch, TAG_NOISE | oi);
            pos += geometric_gap(r.x, op.inv_log);
            if (pos >= len) break;
            apply_hit<T>(t, op, ntgt, (uint32_t)((lo + pos) / W), (uint32_t)((lo + pos) % W),
                         pick_outcome(otab, op.woff, op.nout & 0xFFFF, r.y));
            pos += 1 + geometric_gap(r.z, op.inv_log);
            if (pos >= len) break;
            apply_hit<T>(t, op, ntgt, (uint32_t)((lo + pos) / W), (uint32_t)((lo + pos) % W),
                         pick_outcome(otab, op.woff, op.nout & 0xFFFF, r.w));
            pos++;
        }
    }
}

template <int T>
__device__ __forceinline__ Wd<T> rand_words(const Rng &rng, uint32_t op_i, uint32_t item) {
    uint4 r = rng.draw(item, op_i, TAG_RAND);
    Wd<T> out;
    const uint32_t rs[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
    for (int k = 0; k < T; k++) out.v[k] = rs[k];
    return out;
}

// The items of a Clifford op are independent (no two share a qubit), so that a lane reads the rows of several before it
// writes the first. A lane without a further item repeats its first one: it has read the same rows, and writes the same
// values once more, which costs less than a branch around each item.
template <int T, int NT, uint32_t CODE, int ITEMS>
__device__ __forceinline__ void one_qubit_items(const Tile<T> &t, const uint32_t *w, uint32_t n) {
    for (uint32_t i = threadIdx.x; i < n; i += ITEMS * NT) {
        uint32_t q[ITEMS];
        Wd<T> x[ITEMS], z[ITEMS];
#pragma unroll
        for (int k = 0; k < ITEMS; k++) q[k] = w[i + k * NT < n ? i + k * NT : i];
#pragma unroll
        for (int k = 0; k < ITEMS; k++) {
            x[k] = row<T>(t.X, q[k]);
            z[k] = row<T>(t.Z, q[k]);
        }
#pragma unroll
        for (int k = 0; k < ITEMS; k++) {
            if (CODE == OP_H) {
                row<T>(t.X, q[k]) = z[k];
                row<T>(t.Z, q[k]) = x[k];
            }
            if (CODE == OP_HXY) row<T>(t.Z, q[k]) = wxor(z[k], x[k]);
            if (CODE == OP_HYZ) row<T>(t.X, q[k]) = wxor(x[k], z[k]);
            if (CODE == OP_CXYZ) {
                row<T>(t.X, q[k]) = wxor(x[k], z[k]);
                row<T>(t.Z, q[k]) = x[k];
            }
            if (CODE == OP_CZYX) {
                row<T>(t.X, q[k]) = z[k];
                row<T>(t.Z, q[k]) = wxor(z[k], x[k]);
            }
        }
    }
}
template <int T, int NT, uint32_t CODE>
__device__ __forceinline__ void one_qubit(const Tile<T> &t, const uint32_t *w, uint32_t n) {
    if (T > 2 || n <= NT) one_qubit_items<T, NT, CODE, 1>(t, w, n);
    else if (n <= 2 * NT) one_qubit_items<T, NT, CODE, 2>(t, w, n);
    else one_qubit_items<T, NT, CODE, 4>(t, w, n);
}

template <int T, uint32_t CODE>
__device__ __forceinline__ void two_qubit_rule(Wd<T> &x1, Wd<T> &z1, Wd<T> &x2, Wd<T> &z2) {
    switch (CODE) {
        case OP_CX: z1 = wxor(z1, z2); x2 = wxor(x2, x1); break;
        case OP_CY: z1 = wxor(z1, wxor(x2, z2)); z2 = wxor(z2, x1); x2 = wxor(x2, x1); break;
        case OP_CZ: z1 = wxor(z1, x2); z2 = wxor(z2, x1); break;
        case OP_SWAP: { Wd<T> a = x1; x1 = x2; x2 = a; a = z1; z1 = z2; z2 = a; } break;
        case OP_ISWAP: {
            Wd<T> dx = wxor(x1, x2);
            Wd<T> t1 = wxor(z1, dx), t2 = wxor(z2, dx);
            z1 = t2; z2 = t1;
            Wd<T> a = x1; x1 = x2; x2 = a;
        } break;
        case OP_CXSWAP: z2 = wxor(z2, z1); z1 = wxor(z1, z2); x1 = wxor(x1, x2); x2 = wxor(x2, x1); break;
        case OP_CZSWAP: {
            Wd<T> a = x1; x1 = x2; x2 = a; a = z1; z1 = z2; z2 = a;
            z1 = wxor(z1, x2); z2 = wxor(z2, x1);
        } break;
        case OP_SWAPCX: z1 = wxor(z1, z2); z2 = wxor(z2, z1); x2 = wxor(x2, x1); x1 = wxor(x1, x2); break;
        case OP_SQRTXX: { Wd<T> d = wxor(z1, z2); x1 = wxor(x1, d); x2 = wxor(x2, d); } break;
        case OP_SQRTYY: {
            Wd<T> d = wxor(wxor(x1, z1), wxor(x2, z2));
            x1 = wxor(x1, d); z1 = wxor(z1, d); x2 = wxor(x2, d); z2 = wxor(z2, d);
        } break;
        case OP_SQRTZZ: { Wd<T> d = wxor(x1, x2); z1 = wxor(z1, d); z2 = wxor(z2, d); } break;
        case OP_XCX: x1 = wxor(x1, z2); x2 = wxor(x2, z1); break;
        case OP_XCY: x1 = wxor(x1, wxor(x2, z2)); x2 = wxor(x2, z1); z2 = wxor(z2, z1); break;
        case OP_YCX: x2 = wxor(x2, wxor(x1, z1)); x1 = wxor(x1, z2); z1 = wxor(z1, z2); break;
        case OP_YCY: {
            Wd<T> y1 = wxor(x1, z1), y2 = wxor(x2, z2);
            x1 = wxor(x1, y2); z1 = wxor(z1, y2); x2 = wxor(x2, y1); z2 = wxor(z2, y1);
        } break;
        default: break;
    }
}

template <int T, int NT, uint32_t CODE, int ITEMS>
__device__ __forceinline__ void two_qubit_items(const Tile<T> &t, const uint32_t *w, uint32_t n) {
    for (uint32_t i = threadIdx.x; i < n; i += ITEMS * NT) {
        uint32_t qa[ITEMS], qb[ITEMS];
        Wd<T> x1[ITEMS], z1[ITEMS], x2[ITEMS], z2[ITEMS];
#pragma unroll
        for (int k = 0; k < ITEMS; k++) {
            const uint32_t item = i + k * NT < n ? i + k * NT : i;
            qa[k] = w[2 * item];
            qb[k] = w[2 * item + 1];
        }
#pragma unroll
        for (int k = 0; k < ITEMS; k++) {
            x1[k] = row<T>(t.X, qa[k]);
            z1[k] = row<T>(t.Z, qa[k]);
            x2[k] = row<T>(t.X, qb[k]);
            z2[k] = row<T>(t.Z, qb[k]);
        }
#pragma unroll
        for (int k = 0; k < ITEMS; k++) {
            two_qubit_rule<T, CODE>(x1[k], z1[k], x2[k], z2[k]);
            row<T>(t.X, qa[k]) = x1[k];
            row<T>(t.Z, qa[k]) = z1[k];
            row<T>(t.X, qb[k]) = x2[k];
            row<T>(t.Z, qb[k]) = z2[k];
        }
    }
}
template <int T, int NT, uint32_t CODE>
__device__ __forceinline__ void two_qubit(const Tile<T> &t, const uint32_t *w, uint32_t n) {
    if (T > 2 || n <= NT) two_qubit_items<T, NT, CODE, 1>(t, w, n);
    else two_qubit_items<T, NT, CODE, 2>(t, w, n);
}

// An op's header in scalar registers: all lanes run the same op, so its fields steer scalar branches.
__device__ __forceinline__ DevOp scalar_op(const uint4 &lo, const uint4 &hi) {
    DevOp op;
    op.code = scalar(lo.x);
    op.n = scalar(lo.y);
    op.toff = scalar(lo.z);
    op.base = scalar(lo.w);
    op.p = __uint_as_float(scalar(hi.x));
    op.inv_log = __uint_as_float(scalar(hi.y));
    op.woff = scalar(hi.z);
    op.nout = scalar(hi.w);
    return op;
}

// What bounds it is a tile's chain of dependent steps (compiler.cc, choose_launch, has the launch shapes): a launch of 63
// tiles takes 0.83 of the time of one of 512. So ops are staged a page at a time and not from one barrier to the next
// (5000 qubits, 20 layers: 388 page turns before, 58 with the large pages, and 97 barriers, where ops share rows), and
// steer scalar branches; a lane handles several items of an op at once; and noise keeps its loads in flight while it
// draws. 16384 shots of that circuit 0.548 -> 0.306 ms, of which noise takes 0.10 and the Clifford ops 0.21 (LDS
// transfers alone: 0.07); 1000 shots of the surface code of d = 5 0.110 -> 0.073 ms; 2^18 shots of d = 25 5.06 -> 3.36 ms.
template <int T, int NT>
__global__ __launch_bounds__(NT) void frame_sim_kernel(const uint32_t *__restrict__ blob,
                                                       const uint32_t *__restrict__ ntgt,
                                                       const uint32_t *__restrict__ otab, LaunchParams P) {
    extern __shared__ uint4 lds4[];
    uint32_t *const lds = reinterpret_cast<uint32_t *>(lds4);
    // LDS layout: two staging buffers, then the tile (frame rows, record ring, staged detector rows, observable rows,
    // chain mask).
    Tile<T> t;
    t.X = lds + 2 * P.stage_words;
    t.Z = t.X + P.num_qubits * T;
    t.REC = t.Z + P.num_qubits * T;
    t.STG = t.REC + P.ring * T;
    t.OBS = t.STG + STAGE_ROWS * T;
    t.CHAIN = t.OBS + P.num_obs * T;
    const uint32_t tid = threadIdx.x;
    const uint32_t W = 32 * T;
    const uint64_t shot0 = (uint64_t)blockIdx.x * W;
    const uint64_t tile64 = P.tile0 + blockIdx.x;
    Rng rng{(uint32_t)P.seed, frame_key_hi((uint32_t)(P.seed >> 32), tile64), (uint32_t)tile64};
    const bool randomize = P.randomize != 0;

    for (uint32_t i = tid; i < P.num_qubits; i += NT) {
        row<T>(t.X, i) = wzero<T>();
        row<T>(t.Z, i) = randomize ? rand_words<T>(rng, 0xFFFFFFFFu, i) : wzero<T>();
    }
    for (uint32_t i = tid; i < (P.num_obs + 1) * T; i += NT) t.OBS[i] = 0;
    for (uint32_t i = tid; i < P.page0_len; i += NT) lds[i] = blob[i];
    __syncthreads();

    uint32_t fptr = 0, fend = 0;
    if (P.mode == MODE_FIXED) {
        fptr = P.fault_off[blockIdx.x];
        fend = P.fault_off[blockIdx.x + 1];
    }

    uint32_t buf = 0;
    while (P.page0_len) {
        const uint32_t *cur = lds + buf * P.stage_words;
        const uint4 head = *reinterpret_cast<const uint4 *>(cur);
        const uint32_t n_ops = scalar(head.x), nbeg = scalar(head.y), nlen = scalar(head.z), op0 = scalar(head.w);
        // Prefetch the next page into registers (a lane takes at most two pieces: stage_words <= 8 * NT); it lands in
        // the other staging buffer after this page's ops, so its latency hides behind their work.
        const uint4 *const next = reinterpret_cast<const uint4 *>(blob + nbeg);
        uint4 pre0 = make_uint4(0, 0, 0, 0), pre1 = pre0;
        if (4 * tid < nlen) pre0 = next[tid];
        if (4 * (tid + NT) < nlen) pre1 = next[tid + NT];
        const uint4 *hdrs = reinterpret_cast<const uint4 *>(cur + BLOB_HEADER);
        uint4 next_lo = hdrs[0], next_hi = hdrs[1];

        for (uint32_t j = 0; j < n_ops; j++) {
            const DevOp op = scalar_op(next_lo, next_hi);
            const uint32_t nj = j + 1 < n_ops ? j + 1 : j;
            next_lo = hdrs[2 * nj];
            next_hi = hdrs[2 * nj + 1];
            const uint32_t oi = op0 + j;
            const uint32_t code = op.code & 0xFF;
            const bool rnd = randomize && (op.code & OPF_RANDOMIZE);
            const uint32_t *w = cur + op.toff;
            switch (code) {
                case OP_H: one_qubit<T, NT, OP_H>(t, w, op.n); break;
                case OP_HXY: one_qubit<T, NT, OP_HXY>(t, w, op.n); break;
                case OP_HYZ: one_qubit<T, NT, OP_HYZ>(t, w, op.n); break;
                case OP_CXYZ: one_qubit<T, NT, OP_CXYZ>(t, w, op.n); break;
                case OP_CZYX: one_qubit<T, NT, OP_CZYX>(t, w, op.n); break;
                case OP_CX: two_qubit<T, NT, OP_CX>(t, w, op.n); break;
                case OP_CY: two_qubit<T, NT, OP_CY>(t, w, op.n); break;
                case OP_CZ: two_qubit<T, NT, OP_CZ>(t, w, op.n); break;
                case OP_SWAP: two_qubit<T, NT, OP_SWAP>(t, w, op.n); break;
                case OP_ISWAP: two_qubit<T, NT, OP_ISWAP>(t, w, op.n); break;
                case OP_CXSWAP: two_qubit<T, NT, OP_CXSWAP>(t, w, op.n); break;
                case OP_CZSWAP: two_qubit<T, NT, OP_CZSWAP>(t, w, op.n); break;
                case OP_SWAPCX: two_qubit<T, NT, OP_SWAPCX>(t, w, op.n); break;
                case OP_SQRTXX: two_qubit<T, NT, OP_SQRTXX>(t, w, op.n); break;
                case OP_SQRTYY: two_qubit<T, NT, OP_SQRTYY>(t, w, op.n); break;
                case OP_SQRTZZ: two_qubit<T, NT, OP_SQRTZZ>(t, w, op.n); break;
                case OP_XCX: two_qubit<T, NT, OP_XCX>(t, w, op.n); break;
                case OP_XCY: two_qubit<T, NT, OP_XCY>(t, w, op.n); break;
                case OP_YCX: two_qubit<T, NT, OP_YCX>(t, w, op.n); break;
                case OP_YCY: two_qubit<T, NT, OP_YCY>(t, w, op.n); break;
                case OP_FEEDBACK:
                    for (uint32_t i = tid; i < op.n; i += NT) {
                        const uint32_t slot = w[3 * i], q = w[3 * i + 1], mask = w[3 * i + 2];
                        const Wd<T> r = row<T>(t.REC, slot);
                        if (mask & 1) row<T>(t.X, q) = wxor(row<T>(t.X, q), r);
                        if (mask & 2) row<T>(t.Z, q) = wxor(row<T>(t.Z, q), r);
                    }
                    break;
                case OP_R: case OP_RX: case OP_RY:
                    for (uint32_t i = tid; i < op.n; i += NT) {
                        const uint32_t q = w[i];
                        const Wd<T> r = rnd ? rand_words<T>(rng, oi, i) : wzero<T>();
                        if (code == OP_R) {
                            row<T>(t.X, q) = wzero<T>();
                            if (rnd) row<T>(t.Z, q) = wxor(row<T>(t.Z, q), r);
                        } else if (code == OP_RX) {
                            row<T>(t.Z, q) = wzero<T>();
                            if (rnd) row<T>(t.X, q) = wxor(row<T>(t.X, q), r);
                        } else {
                            Wd<T> z = rnd ? wxor(row<T>(t.Z, q), r) : row<T>(t.Z, q);
                            row<T>(t.Z, q) = z;
                            row<T>(t.X, q) = z;
                        }
                    }
                    break;
                case OP_M: case OP_MX: case OP_MY: case OP_MR: case OP_MRX: case OP_MRY:
                    for (uint32_t i = tid; i < op.n; i += NT) {
                        const uint32_t q = w[i];
                        Wd<T> x = row<T>(t.X, q), z = row<T>(t.Z, q);
                        const Wd<T> r = rnd ? rand_words<T>(rng, oi, i) : wzero<T>();
                        Wd<T> rec;
                        if (code == OP_M || code == OP_MR) {
                            rec = x;
                            if (code == OP_MR) x = wzero<T>();
                            z = wxor(z, r);
                        } else if (code == OP_MX || code == OP_MRX) {
                            rec = z;
                            if (code == OP_MRX) z = wzero<T>();
                            x = wxor(x, r);
                        } else {
                            rec = wxor(x, z);
                            if (code == OP_MY) {
                                x = wxor(x, r);
                                z = wxor(z, r);
                            } else {
                                z = wxor(z, r);
                                x = z;
                            }
                        }
                        row<T>(t.X, q) = x;
                        row<T>(t.Z, q) = z;
                        row<T>(t.REC, op.base + i) = rec;
                    }
                    break;
                case OP_MPP:
                case OP_SPP:
                    for (uint32_t i = tid; i < op.n; i += NT) {
                        const uint32_t b = w[i], e2 = w[i + 1];
                        Wd<T> v = wzero<T>();
                        for (uint32_t k = b; k < e2; k++) {
                            const uint32_t term = w[k];
                            if (term & TERM_PAULI) {
                                const uint32_t q = term & TERM_QMASK;
                                if (term & TERM_X) v = wxor(v, row<T>(t.Z, q));
                                if (term & TERM_Z) v = wxor(v, row<T>(t.X, q));
                            } else {
                                v = wxor(v, row<T>(t.REC, term));
                            }
                        }
                        Wd<T> apply;
                        if (code == OP_MPP) {
                            row<T>(t.REC, op.base + i) = v;
                            if (!rnd) continue;
                            apply = rand_words<T>(rng, oi, i);
                        } else {
                            apply = v;
                        }
                        for (uint32_t k = b; k < e2; k++) {
                            const uint32_t term = w[k];
                            if (!(term & TERM_PAULI)) continue;
                            const uint32_t q = term & TERM_QMASK;
                            if (term & TERM_X) row<T>(t.X, q) = wxor(row<T>(t.X, q), apply);
                            if (term & TERM_Z) row<T>(t.Z, q) = wxor(row<T>(t.Z, q), apply);
                        }
                    }
                    break;
                case OP_RECZERO:
                    for (uint32_t i = tid; i < op.n; i += NT) row<T>(t.REC, op.base + i) = wzero<T>();
                    break;
                case OP_DET:
                    for (uint32_t i = tid; i < op.n; i += NT) {
                        const uint32_t b = w[i], e2 = w[i + 1];
                        Wd<T> v = wzero<T>();
                        for (uint32_t k = b; k < e2; k++) v = wxor(v, row<T>(t.REC, w[k]));
                        if (P.det_invert) {
                            const uint32_t d = op.base + i;
                            if ((P.det_invert[d >> 5] >> (d & 31)) & 1u) {
#pragma unroll
                                for (int k = 0; k < T; k++) v.v[k] = ~v.v[k];
                            }
                        }
                        row<T>(t.STG, (op.base + i) % STAGE_ROWS) = v;
                    }
                    break;
                case OP_OBS:
                    for (uint32_t i = tid; i < op.n; i += NT) {
                        const uint32_t b = w[i], e2 = w[i + 1];
                        const uint32_t idx = w[b];
                        Wd<T> v = wzero<T>();
                        for (uint32_t k = b + 1; k < e2; k++) {
                            const uint32_t term = w[k];
                            if (term & TERM_PAULI) {
                                const uint32_t q = term & TERM_QMASK;
                                if (term & TERM_X) v = wxor(v, row<T>(t.Z, q));
                                if (term & TERM_Z) v = wxor(v, row<T>(t.X, q));
                            } else {
                                v = wxor(v, row<T>(t.REC, term));
                            }
                        }
#pragma unroll
                        for (int k = 0; k < T; k++) {
                            if (v.v[k]) atomicXor(&t.OBS[idx * T + k], v.v[k]);
                        }
                    }
                    break;
                case OP_FLUSH:
                    if (P.dets.enabled) flush_rows<T, NT>(t.STG, op.n, op.base, P.dets, shot0, P.shots);
                    break;
                case OP_FLUSH_OBS:
                    if (P.obs.enabled) flush_rows<T, NT>(t.OBS, op.n, 0, P.obs, shot0, P.shots);
                    break;
                case OP_CHAINCLR:
                    if (tid < T) t.CHAIN[tid] = 0;
                    break;
                case OP_NOISE1: case OP_NOISE2: case OP_MFLIP: case OP_CORR: case OP_HERALD: {
                    if (P.mode == MODE_FIXED) {
                        // Faults of this tile are sorted by op; consume the prefix that belongs to this op.
                        while (true) {
                            const uint32_t idx = fptr + tid;
                            bool mine = false;
                            if (idx < fend) {
                                const DevFault f = P.faults[idx];
                                if (f.op == oi) {
                                    mine = true;
                                    apply_hit<T>(t, op, ntgt, f.site, f.shot, f.code);
                                }
                            }
                            const uint32_t cnt = __syncthreads_count(mine);
                            fptr += cnt;
                            if (cnt < NT) break;
                        }
                        break;
                    }
                    if (P.mode != MODE_SAMPLED || !(op.p > 0.0f)) break;
                    const uint32_t nout = op.nout & 0xFFFF;
                    if (op.code & OPF_DENSE) {
                        // Dense draw: Bernoulli word per (site, word), then one outcome per fired shot.
                        for (uint32_t i = tid; i < op.n * T; i += NT) {
                            const uint32_t site = i / T, wd = i % T;
                            uint32_t fire = bernoulli_word(op.p, rng, i, oi);
                            uint32_t ctr = 0;
                            uint4 r = make_uint4(0, 0, 0, 0);
                            while (fire) {
                                const uint32_t b = __ffs(fire) - 1;
                                fire &= fire - 1;
                                if ((ctr & 3) == 0) r = rng.draw(i, 0x40000000u | ctr, TAG_NOISE | oi);
                                const uint32_t rs = (ctr & 3) == 0 ? r.x : (ctr & 3) == 1 ? r.y : (ctr & 3) == 2 ? r.z : r.w;
                                ctr++;
                                apply_hit<T>(t, op, ntgt, site, wd * 32 + b, pick_outcome(otab, op.woff, nout, rs));
                            }
                        }
                        break;
                    }
                    const uint64_t N = (uint64_t)op.n * W;
                    // Chunks of 64 positions or more, up to 2^(cmax + 2), so that there are at most 2^chunk_log of them if that allows it.
                    const uint32_t cmax = (op.nout >> 16) & 0xFF;
                    const uint64_t each = (N + (1u << P.chunk_log) - 1) >> P.chunk_log;
                    const uint32_t clog = min(cmax + 2, max(6u, each > 1 ? 64u - (uint32_t)__clzll(each - 1) : 0u));
                    if (code == OP_NOISE1) {
                        sparse_noise<T, NT, OP_NOISE1>(t, op, ntgt, otab, rng, oi, clog, N);
                    } else if (code == OP_NOISE2) {
                        sparse_noise<T, NT, OP_NOISE2>(t, op, ntgt, otab, rng, oi, clog, N);
                    } else if (code == OP_MFLIP) {
                        sparse_noise<T, NT, OP_MFLIP>(t, op, ntgt, otab, rng, oi, clog, N);
                    } else if (code == OP_HERALD) {
                        sparse_noise<T, NT, OP_HERALD>(t, op, ntgt, otab, rng, oi, clog, N);
                    } else {
                        sparse_chain<T, NT>(t, op, ntgt, otab, rng, oi, clog, N);
                    }
                    break;
                }
                default:
                    break;
            }
            // The last op of a page has the page turn's barrier.
            if ((op.code & OPF_SYNC) && j + 1 < n_ops) __syncthreads();
        }
        if (nlen == 0) break;
        uint4 *nst = reinterpret_cast<uint4 *>(lds + (buf ^ 1) * P.stage_words);
        if (4 * tid < nlen) nst[tid] = pre0;
        if (4 * (tid + NT) < nlen) nst[tid + NT] = pre1;
        __syncthreads();
        buf ^= 1;
    }
}

__global__ void pack_rows_kernel(const uint8_t *src, size_t src_stride, uint8_t *dst, size_t dst_stride,
                                 uint64_t rows, uint32_t ncols) {
    const uint32_t nb = (ncols + 7) / 8;
    const uint64_t total = rows * nb;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t r = i / nb;
        const uint32_t c = (uint32_t)(i % nb);
        uint32_t v = 0;
        for (uint32_t b = 0; b < 8; b++) {
            const uint32_t col = 8 * c + b;
            if (col < ncols) v |= (uint32_t)(src[r * src_stride + col] & 1u) << b;
        }
        dst[r * dst_stride + c] = (uint8_t)v;
    }
}

}  // namespace

// Host-side launcher (C++ linkage, called from sampler.cc).
namespace sa {

hipError_t launch_frame_kernel(int T, const DevProgram &prog, const LaunchParams &P, uint32_t num_tiles, size_t lds,
                               uint32_t lanes, hipStream_t stream) {
    if (num_tiles == 0) return hipSuccess;
    if (P.stage_words > 8 * lanes) return hipErrorInvalidValue;
#define STIM_AMD_LAUNCH(TW, NB)                                                                                   \
    if (T == TW && lanes == NB) {                                                                                 \
        static size_t reserved = 0;                                                                               \
        const hipError_t e = reserve_lds((const void *)frame_sim_kernel<TW, NB>, lds, reserved);                  \
        if (e != hipSuccess) return e;                                                                            \
        hipLaunchKernelGGL((frame_sim_kernel<TW, NB>), dim3(num_tiles), dim3(NB), lds, stream, prog.blob,         \
                           prog.ntgt, prog.otab, P);                                                              \
        return hipGetLastError();                                                                                 \
    }
    STIM_AMD_LAUNCH(1, 256)
    STIM_AMD_LAUNCH(1, 512)
    STIM_AMD_LAUNCH(1, 1024)
    STIM_AMD_LAUNCH(2, 256)
    STIM_AMD_LAUNCH(2, 512)
    STIM_AMD_LAUNCH(2, 1024)
    STIM_AMD_LAUNCH(4, 256)
    STIM_AMD_LAUNCH(4, 512)
    STIM_AMD_LAUNCH(4, 1024)
#undef STIM_AMD_LAUNCH
    return hipErrorInvalidValue;
}

hipError_t launch_pack_rows(const uint8_t *src, size_t src_stride, uint8_t *dst, size_t dst_stride, uint64_t rows,
                            uint32_t ncols, hipStream_t stream) {
    const uint64_t total = rows * ((ncols + 7) / 8);
    if (total == 0) return hipSuccess;
    const uint32_t blocks = (uint32_t)std::min<uint64_t>((total + 255) / 256, 65536);
    hipLaunchKernelGGL(pack_rows_kernel, dim3(blocks), dim3(256), 0, stream, src, src_stride, dst, dst_stride, rows, ncols);
    return hipGetLastError();
}

}  // namespace sa

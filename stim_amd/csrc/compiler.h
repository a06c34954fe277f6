// Lowers a flattened circuit into the device program executed by the frame kernel.
#pragma once

#include <cstdint>
#include <vector>

#include "circuit.h"
#include "program.h"

namespace sa {

// Where the sites of one flat instruction landed in the device program (one entry per emitted
// noise op; an instruction split into segments has several entries).
struct SiteRange {
    uint32_t op;        // device op index
    uint32_t first;     // first site (group index within the instruction) covered by the op
    uint32_t count;     // sites covered
};

// The ops packed into pages for staging buffers of stage_words words.
struct PageSet {
    uint32_t stage_words = OP_STAGE_WORDS;
    size_t at = 0;          // word of Program::blob at which the first page starts
    uint32_t page0_len = 0; // its words
};

struct Program {
    std::vector<DevOp> ops;
    std::vector<uint32_t> tgt;    // frame-op words (before packing into pages)
    std::vector<uint32_t> blob;   // pages (program.h layout) as the device walks them, of both sets
    PageSet small, large;         // the smallest staging buffers; the largest that help (choose_launch)
    std::vector<uint32_t> ntgt;   // noise-op words
    std::vector<uint32_t> otab;
    uint32_t num_qubits = 0;      // dense qubit rows
    uint32_t ring = 1;            // record ring rows
    uint32_t num_detectors = 0;
    uint32_t num_observables = 0;
    uint64_t num_measurements = 0;
    uint32_t num_noise_ops = 0;
    uint32_t num_syncs = 0;
    bool has_randomizing_ops = false;
    // flat instruction index -> site ranges of its noise ops
    std::vector<std::vector<SiteRange>> sites;
    Stats stats;
};

// measurement_outputs: the outputs are the circuit's measurement results in record order (one
// output row per result) instead of its detectors and observables.
Program compile_program(const std::vector<const Instr *> &flat, bool measurement_outputs = false);

// Resolves a fault (flat instruction index, group index, code) to (op, site); throws
// std::out_of_range when the instruction has no such noise site.
void resolve_fault(const Program &prog, uint32_t k, uint32_t j, uint32_t *op, uint32_t *site);

// A tile has two words per row (64 shots) up to this figure of tile_bytes, else one.
constexpr size_t FRAME_T2_BYTES = 64 * 1024;
// LDS bytes of a tile of 32*T shots with the smallest staging buffers. Tile widths, what fits, and the lanes that
// noise is cut for go by this figure: they fix the random streams.
size_t tile_bytes(const Program &prog, int T);

// How the frame kernel is launched for a number of tiles of 32*T shots.
struct FrameLaunch {
    const PageSet *pages;
    size_t lds;
    uint32_t lanes;
};
FrameLaunch choose_launch(const Program &prog, int T, uint64_t tiles);

}  // namespace sa

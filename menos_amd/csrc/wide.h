// Passes of dense blocks wider than a window pass takes (wide.hip).
#pragma once

#include <cstdint>
#include <vector>

#include "mh_internal.h"

namespace mh {

// Tile qubits of a wide pass: the smallest state it takes.
constexpr uint32_t kWideTileBits = 12;
// ... and the largest: a workgroup of 512 threads a tile, and a launch takes
// fewer than 2^32 threads (a complex64 state of 35 qubits, 256 GiB, goes to the
// per-group kernel, whose grid does not grow with it).
constexpr uint32_t kWideQubits = 34;
// Blocks of one pass at most: its arithmetic is by then many times the read
// and write of the state that they share, and a run's monitor is asked between
// passes.
constexpr uint32_t kWidePassBlocks = 16;

// Tables of one upload, about (a run with a budget keeps to what that leaves).
constexpr uint64_t kWideTableBytes = uint64_t{16} << 20;

// Whether a dense block of k qubits of an n-qubit state goes to a wide pass:
// three to six qubits, except the complex64 blocks that the matrix cores take
// and states beyond one launch.
bool wide_applies(int32_t precision, uint32_t n, uint32_t k);

// Device bytes of the tables of any one pass of these blocks, at most.
uint64_t wide_pass_bytes(int32_t precision, uint32_t n, const std::vector<Block>& blocks);

// The lowest qubits, which every tile holds: runs of 128 bytes.
uint64_t wide_low_mask(int32_t precision);

// Tables of passes over one state, each of consecutive wide blocks whose
// operands and low run fit a tile; add() on the host, then upload(), then
// launches in any order.
class WidePasses {
public:
    WidePasses(uint32_t n, int32_t precision);
    ~WidePasses();
    WidePasses(const WidePasses&) = delete;
    WidePasses& operator=(const WidePasses&) = delete;
    // Returns the pass's index.
    uint32_t add(const std::vector<Block>& blocks, const std::vector<uint32_t>& which);
    uint64_t bytes() const;
    // What add() would add to them, at most.
    uint64_t bytes_of(const std::vector<Block>& blocks, const std::vector<uint32_t>& which) const;
    void upload();
    void launch(void* state, uint32_t pass, hipStream_t stream) const;

private:
    struct Impl;
    Impl* impl_;
};

}  // namespace mh

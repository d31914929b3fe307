// Dense blocks of three to six qubits, several to a pass over the state.
//
// A workgroup takes 2^12 amplitudes (the tile bits T: the operands of the
// pass's blocks, the lowest qubits for whole 128-byte runs, then the next
// lowest) into LDS, applies the blocks there one after another, and writes
// them back, so blocks that share a pass share one read and write of the
// state. The arithmetic is the per-group kernel's (gates.hip), operation by
// operation: every output starts at (+0, +0) and adds M[out][in] * a[in] for
// in ascending, so complex128 results are the reference CPU generic kernel's
// bits (reference src/kernels/cpu/dense_kernels.cpp:465-524).
//
// What bounds it: a block of k qubits takes 2^k * 8 operations in double an
// amplitude (none fused, for the bits), which at four cycles a wavefront is 55,
// 109, 218 us for k = 3, 4, 5 at 25 qubits against 195 us for the read and
// write. So the split keeps every SIMD on that arithmetic for every k: a thread
// computes eight outputs of a group, with 2^(k-3) threads (of different
// wavefronts) sharing a group, each input read from LDS once for them and the
// matrix column for the eight brought in by scalar loads. One thread per group
// of 2^k amplitudes held them all in registers (64 to 256 of them), left few
// wavefronts to hide the loads, and each block read and wrote the state.
//
// A call at 25 qubits complex128, before and now: one block of k = 3, 4, 5, 6:
// 0.28, 0.36, 0.96, 6.04 -> 0.22, 0.24, 0.33, 0.69 ms; three blocks (3, 3, 4)
// and (3, 5, 3): 0.92, 1.49 -> 0.36, 0.62 ms. complex64, one block of k = 3, 4:
// 0.114, 0.177 -> 0.099, 0.111 ms; (3, 3, 4) 0.38 -> 0.17 ms. A grid of resident
// workgroups that takes the next tile to registers meanwhile was slower
// throughout (0.31 ms for k = 3): the loads then wait behind the stores.
#include <algorithm>
#include <cstring>

#include "wide.h"

namespace mh {
namespace {

constexpr uint32_t kTileBits = kWideTileBits;
constexpr uint32_t kThreads = 512;
constexpr uint32_t kOuts = (1u << kTileBits) / kThreads;  // outputs (and loaded amplitudes) of a thread
constexpr uint32_t kThreadBits = 9;
constexpr uint32_t kMaxK = 6;
static_assert(kOuts == 8 && kThreads == 1u << kThreadBits);
static_assert((uint64_t{1} << (kWideQubits - kTileBits)) * kThreads < uint64_t{1} << 32);

template <typename R> struct Vec;
template <> struct Vec<double> { using type = double2; };
template <> struct Vec<float> { using type = float2; };

// One block on the tile. Amplitude e of the tile lies at place(e).
struct WideBlock {
    uint32_t k;
    uint32_t mat;                       // its matrix: entry [sub][in][8] from here (complex numbers)
    uint32_t sorted[kMaxK];             // operands' tile bits, ascending
    uint32_t member[1u << kMaxK];       // byte offset of member l (operand j set where bit j of l is)
    uint32_t moves;                     // the matrix permutes the basis: no arithmetic but its zeros'
    uint32_t source[1u << kMaxK];       // ... byte offset of the member that output l takes
};

struct WideArgs {
    void* state;
    const WideBlock* blocks;
    const void* mats;
    uint64_t outer_mask;                // index bits outside T: the tile index deposits here, ascending
    uint32_t count;
    uint32_t pad;
    uint8_t tpos[16];                   // tile bit i -> qubit, ascending
};

// The tables are read-only while a pass runs: through the constant address
// space they come in by scalar loads.
#define MH_CONSTANT __attribute__((address_space(4)))
template <typename R> using Entry = R __attribute__((ext_vector_type(2)));
template <typename R> using EntryPtr = const MH_CONSTANT Entry<R>*;
typedef const MH_CONSTANT WideBlock* BlockPtr;

// Where amplitude e of a tile lies (in amplitudes): the low three bits take the
// sum of e's four groups of three, so that lanes whose amplitudes are 8, 64 or
// 512 apart (a block on the lowest tile bits) use different banks. Linear over
// XOR.
__host__ __device__ constexpr uint32_t place(uint32_t e) { return e ^ (((e >> 3) ^ (e >> 6) ^ (e >> 9)) & 7u); }

__device__ __forceinline__ void cmac(double& sr, double& si, double mr, double mi, double ar, double ai) {
    const double pr = mr * ar - mi * ai;
    const double pi = mr * ai + mi * ar;
    sr = sr + pr;
    si = si + pi;
}

__device__ __forceinline__ void cmac(float& sr, float& si, float mr, float mi, float ar, float ai) {
    sr = __builtin_fmaf(mr, ar, sr);
    sr = __builtin_fmaf(-mi, ai, sr);
    si = __builtin_fmaf(mr, ai, si);
    si = __builtin_fmaf(mi, ar, si);
}

template <typename R, uint32_t K>
__device__ __forceinline__ void apply(unsigned char* lds, BlockPtr blk, EntryPtr<R> mats, uint32_t t) {
    using V = typename Vec<R>::type;
    constexpr uint32_t dim = 1u << K;
    const uint32_t sub = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(t >> (kTileBits - K))));
    uint32_t base = t & ((1u << (kTileBits - K)) - 1u);
#pragma unroll
    for (uint32_t j = 0; j < K; ++j) {
        const uint32_t low = (1u << blk->sorted[j]) - 1u;
        base = ((base & ~low) << 1) | (base & low);
    }
    const uint32_t from = place(base) * sizeof(V);
    const EntryPtr<R> m = mats + blk->mat + sub * (dim * kOuts);
    R sr[kOuts], si[kOuts];
#pragma unroll
    for (uint32_t o = 0; o < kOuts; ++o) sr[o] = si[o] = R(0);
    // One input at a time: unrolled, the scalar loads of wide blocks' matrices
    // (16 KB for k = 5, as much as the scalar cache) wait on each other (0.69
    // against 0.88 ms for k = 6 at 25 qubits, the same for k = 3 and 4).
#pragma unroll 1
    for (uint32_t in = 0; in < dim; ++in) {
        const V a = *reinterpret_cast<const V*>(lds + (from ^ blk->member[in]));
#pragma unroll
        for (uint32_t o = 0; o < kOuts; ++o) {
            const Entry<R> e = m[in * kOuts + o];
            cmac(sr[o], si[o], e[0], e[1], a.x, a.y);
        }
    }
    if constexpr (K > 3) __syncthreads();  // the group's other threads have read it
#pragma unroll
    for (uint32_t o = 0; o < kOuts; ++o) {
        V r;
        r.x = sr[o];
        r.y = si[o];
        *reinterpret_cast<V*>(lds + (from ^ blk->member[sub * kOuts + o])) = r;
    }
    __syncthreads();
}

// A block that permutes the basis (a Toffoli, a controlled SWAP): its sums are
// one product by 1 and products by 0, so an output is its source plus the sum
// of every input times zero: +0 where they are finite; where one is not, the
// group turns NaN, as its sums would (but for the part of an infinity moved). Beside 8 * 2^k operations an amplitude it
// costs nothing: 24 blocks at 25 qubits, half of them Toffolis, 3.10 -> 2.55 ms.
template <typename R, uint32_t K>
__device__ __forceinline__ void permute(unsigned char* lds, BlockPtr blk, uint32_t t) {
    using V = typename Vec<R>::type;
    constexpr uint32_t dim = 1u << K;
    const uint32_t sub = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(t >> (kTileBits - K))));
    uint32_t base = t & ((1u << (kTileBits - K)) - 1u);
#pragma unroll
    for (uint32_t j = 0; j < K; ++j) {
        const uint32_t low = (1u << blk->sorted[j]) - 1u;
        base = ((base & ~low) << 1) | (base & low);
    }
    const uint32_t from = place(base) * sizeof(V);
    R zero = R(0);
#pragma unroll 8
    for (uint32_t in = 0; in < dim; ++in) {
        const V a = *reinterpret_cast<const V*>(lds + (from ^ blk->member[in]));
        zero = zero + a.x * R(0);
        zero = zero + a.y * R(0);
    }
    V out[kOuts];
#pragma unroll
    for (uint32_t o = 0; o < kOuts; ++o) {
        const V a = *reinterpret_cast<const V*>(lds + (from ^ blk->source[sub * kOuts + o]));
        out[o].x = a.x + zero;
        out[o].y = a.y + zero;
    }
    if constexpr (K > 3) __syncthreads();  // the group's other threads have read it
#pragma unroll
    for (uint32_t o = 0; o < kOuts; ++o)
        *reinterpret_cast<V*>(lds + (from ^ blk->member[sub * kOuts + o])) = out[o];
    __syncthreads();
}

template <typename R, uint32_t K>
__device__ __forceinline__ void block(unsigned char* lds, BlockPtr blk, EntryPtr<R> mats, uint32_t t) {
    if (blk->moves)
        permute<R, K>(lds, blk, t);
    else
        apply<R, K>(lds, blk, mats, t);
}

template <typename R>
__global__ void __launch_bounds__(kThreads, 4) wide_kernel(WideArgs args) {
    using V = typename Vec<R>::type;
    __shared__ __align__(16) unsigned char lds[sizeof(V) << kTileBits];
    V* const tile = reinterpret_cast<V*>(lds);
    const uint32_t t = threadIdx.x;
    uint64_t at = 0, step[3];
#pragma unroll
    for (uint32_t i = 0; i < kThreadBits; ++i) at |= uint64_t((t >> i) & 1u) << args.tpos[i];
#pragma unroll
    for (uint32_t i = 0; i < 3; ++i) step[i] = 1ull << args.tpos[kThreadBits + i];
    uint64_t outer = 0, om = args.outer_mask;
    for (uint32_t v = blockIdx.x; v != 0; v >>= 1) {
        const uint64_t low = om & (~om + 1);
        if (v & 1u) outer |= low;
        om ^= low;
    }
    V* const s = static_cast<V*>(args.state) + outer + at;
    V v[kOuts];
#pragma unroll
    for (uint32_t r = 0; r < kOuts; ++r)
        v[r] = s[((r & 1u) ? step[0] : 0) + ((r & 2u) ? step[1] : 0) + ((r & 4u) ? step[2] : 0)];
#pragma unroll
    for (uint32_t r = 0; r < kOuts; ++r) tile[place(r * kThreads + t)] = v[r];
    __syncthreads();
    const BlockPtr blocks = (BlockPtr)args.blocks;
    const EntryPtr<R> mats = (EntryPtr<R>)args.mats;
    for (uint32_t b = 0; b < args.count; ++b) {
        const BlockPtr blk = blocks + b;
        switch (blk->k) {
            case 3: block<R, 3>(lds, blk, mats, t); break;
            case 4: block<R, 4>(lds, blk, mats, t); break;
            case 5: block<R, 5>(lds, blk, mats, t); break;
            default: block<R, 6>(lds, blk, mats, t); break;
        }
    }
#pragma unroll
    for (uint32_t r = 0; r < kOuts; ++r)
        s[((r & 1u) ? step[0] : 0) + ((r & 2u) ? step[1] : 0) + ((r & 4u) ? step[2] : 0)] = tile[place(r * kThreads + t)];
}

}  // namespace

bool wide_applies(int32_t precision, uint32_t n, uint32_t k) {
    return n >= kWideTileBits && n <= kWideQubits && k >= 3 && k <= (precision == MH_C128 ? kMaxK : 4);
}

uint64_t wide_pass_bytes(int32_t precision, uint32_t n, const std::vector<Block>& blocks) {
    uint64_t sum = 0, most = 0;
    for (const Block& b : blocks) {
        if (b.diagonal || !wide_applies(precision, n, static_cast<uint32_t>(b.operands.size()))) continue;
        const uint64_t bytes = sizeof(WideBlock) + b.matrix.size() * amp_bytes(precision);
        sum += bytes;
        most = std::max(most, bytes);
    }
    return sum == 0 ? 0 : std::min(sum, kWidePassBlocks * most) + 256;
}

uint64_t wide_low_mask(int32_t precision) { return precision == MH_C128 ? 7 : 15; }

struct WidePasses::Impl {
    struct Pass {
        uint64_t outer_mask;
        uint32_t first, count;
        uint8_t tpos[16];
    };
    uint32_t n;
    int32_t precision;
    std::vector<Pass> passes;
    std::vector<WideBlock> blocks;
    std::vector<double2> mats;
    std::vector<float2> mats32;
    std::vector<unsigned char> host;  // the copy's source, for as long as the device's
    DeviceBuffer tables;              // the blocks, then the matrices
    uint64_t mats_at = 0;
};

WidePasses::WidePasses(uint32_t n, int32_t precision) : impl_(new Impl) {
    impl_->n = n;
    impl_->precision = precision;
}

WidePasses::~WidePasses() { delete impl_; }

uint32_t WidePasses::add(const std::vector<Block>& blocks, const std::vector<uint32_t>& which) {
    Impl& d = *impl_;
    const uint32_t n = d.n;
    uint64_t tile = wide_low_mask(d.precision);
    for (uint32_t b : which) {
        const uint32_t k = static_cast<uint32_t>(blocks[b].operands.size());
        if (!wide_applies(d.precision, n, k)) fail(MH_ERR_INTERNAL, "wide pass: block width out of range");
        uint64_t own = 0;
        for (uint32_t q : blocks[b].operands) {
            if (q >= n || ((own >> q) & 1u)) fail(MH_ERR_INTERNAL, "wide pass: operands out of range or repeated");
            own |= uint64_t{1} << q;
        }
        tile |= own;
    }
    if (static_cast<uint32_t>(__builtin_popcountll(tile)) > kTileBits)
        fail(MH_ERR_INTERNAL, "wide pass: the blocks do not fit a tile");
    for (uint32_t q = 0; static_cast<uint32_t>(__builtin_popcountll(tile)) < kTileBits; ++q) tile |= uint64_t{1} << q;
    Impl::Pass pass{};
    pass.outer_mask = ((uint64_t{1} << n) - 1) & ~tile;
    pass.first = static_cast<uint32_t>(d.blocks.size());
    pass.count = static_cast<uint32_t>(which.size());
    uint32_t bit_of[64] = {};
    for (uint32_t q = 0, i = 0; q < n; ++q)
        if ((tile >> q) & 1u) {
            bit_of[q] = i;
            pass.tpos[i++] = static_cast<uint8_t>(q);
        }
    const bool wide = d.precision == MH_C128;
    for (uint32_t b : which) {
        const Block& blk = blocks[b];
        WideBlock w{};
        w.k = static_cast<uint32_t>(blk.operands.size());
        const uint32_t dim = 1u << w.k;
        w.mat = static_cast<uint32_t>(wide ? d.mats.size() : d.mats32.size());
        for (uint32_t j = 0; j < w.k; ++j) w.sorted[j] = bit_of[blk.operands[j]];
        std::sort(w.sorted, w.sorted + w.k);
        for (uint32_t l = 0; l < dim; ++l) {
            uint32_t e = 0;
            for (uint32_t j = 0; j < w.k; ++j)
                if ((l >> j) & 1u) e |= 1u << bit_of[blk.operands[j]];
            w.member[l] = place(e) * static_cast<uint32_t>(wide ? sizeof(double2) : sizeof(float2));
        }
        // Its source for each output, if the matrix is one 1 to a row and else 0.
        w.moves = 1;
        for (uint32_t o = 0; o < dim; ++o) {
            uint32_t ones = 0;
            for (uint32_t in = 0; in < dim; ++in) {
                const cplx m = blk.matrix[std::size_t(o) * dim + in];
                if (m == cplx(1.0, 0.0)) {
                    ++ones;
                    w.source[o] = w.member[in];
                } else if (m != cplx(0.0, 0.0)) {
                    ones = 2;
                }
            }
            if (ones != 1) w.moves = 0;
        }
        if (w.moves) {
            d.blocks.push_back(w);
            continue;
        }
        for (uint32_t sub = 0; sub < dim / kOuts; ++sub)
            for (uint32_t in = 0; in < dim; ++in)
                for (uint32_t o = 0; o < kOuts; ++o) {
                    const cplx m = blk.matrix[std::size_t(sub * kOuts + o) * dim + in];
                    if (wide)
                        d.mats.push_back(make_double2(m.real(), m.imag()));
                    else
                        d.mats32.push_back(make_float2(static_cast<float>(m.real()), static_cast<float>(m.imag())));
                }
        d.blocks.push_back(w);
    }
    d.passes.push_back(pass);
    return static_cast<uint32_t>(d.passes.size() - 1);
}

uint64_t WidePasses::bytes_of(const std::vector<Block>& blocks, const std::vector<uint32_t>& which) const {
    uint64_t sum = 0;
    for (uint32_t b : which) sum += sizeof(WideBlock) + blocks[b].matrix.size() * amp_bytes(impl_->precision);
    return sum;
}

uint64_t WidePasses::bytes() const {
    return impl_->blocks.size() * sizeof(WideBlock) + impl_->mats.size() * sizeof(double2) +
           impl_->mats32.size() * sizeof(float2);
}

void WidePasses::upload() {
    Impl& d = *impl_;
    const bool wide = d.precision == MH_C128;
    const void* m = wide ? static_cast<const void*>(d.mats.data()) : d.mats32.data();
    const std::size_t bytes = wide ? d.mats.size() * sizeof(double2) : d.mats32.size() * sizeof(float2);
    d.mats_at = (d.blocks.size() * sizeof(WideBlock) + 255) / 256 * 256;
    d.host.resize(d.mats_at + bytes);
    std::memcpy(d.host.data(), d.blocks.data(), d.blocks.size() * sizeof(WideBlock));
    if (bytes > 0) std::memcpy(d.host.data() + d.mats_at, m, bytes);
    d.tables = DeviceBuffer(d.host.size());
    mh::upload(d.tables.get(), d.host.data(), d.host.size());
}

void WidePasses::launch(void* state, uint32_t pass, hipStream_t stream) const {
    const Impl& d = *impl_;
    const Impl::Pass& p = d.passes[pass];
    WideArgs a{};
    a.state = state;
    a.blocks = d.tables.as<WideBlock>() + p.first;
    a.mats = d.tables.as<unsigned char>() + d.mats_at;
    a.outer_mask = p.outer_mask;
    a.count = p.count;
    std::memcpy(a.tpos, p.tpos, sizeof(a.tpos));
    if (d.n < kTileBits || d.n > kWideQubits) fail(MH_ERR_INTERNAL, "wide pass shape out of range");
    const uint32_t tiles = 1u << (d.n - kTileBits);
    if (d.precision == MH_C128)
        hipLaunchKernelGGL(wide_kernel<double>, dim3(tiles), dim3(kThreads), 0, stream, a);
    else
        hipLaunchKernelGGL(wide_kernel<float>, dim3(tiles), dim3(kThreads), 0, stream, a);
    MH_HIP(hipGetLastError());
}

}  // namespace mh

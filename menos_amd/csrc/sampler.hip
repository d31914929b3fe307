// Exact shot sampling on the device.
//
// The reference sampler (src/engines/dense/sample.cpp:24-75) walks the basis in
// index order with `c = fl(c + p_i)`, p_i = x_i*x_i + y_i*y_i (std::norm, no
// FMA), and sends each sorted uniform u to the first basis with u < c (the last
// basis if none). Counts must be identical, so the device reproduces that
// rounding chain bit for bit, in parallel:
//
//  * While c stays in one binade it is an integer multiple K of ulp = 2^s
//    (s = max(exponent(c) - 52, -1074)), and fl(K*2^s + p) = (K + r)*2^s with
//    r = p / 2^s rounded to the nearest integer, ties going to the r that
//    makes K + r even. So a run of steps is an integer sum whose only state is
//    the parity of K: each element is a function of that parity, and these
//    functions compose associatively (exact integer arithmetic, any order).
//  * The binade each block of 2^13 elements (2^11 for states of at most 20
//    qubits) starts in is guessed as if every basis were as likely, and the
//    block's transfer in it is found in the same read of the state as its FP64
//    sum. The prefix of those sums predicts the binade better: blocks guessed
//    wrong are read again. Each 256 blocks' transfers are composed in parallel.
//  * One workgroup then follows the chain: a parallel scan of up to 256
//    transfers gives the exact value after each of them up to the first that
//    does not apply (the running value is not in the predicted binade, or
//    leaves it). There the chain goes on inside: a group's blocks, or a
//    block's elements.
//  * Inside a block the same scan runs over 256 runs of up to eight elements;
//    the run that leaves the binade is walked with plain FP64 adds, and the
//    scan goes on behind it in the next binade (exact_stage).
//  * One workgroup per block that holds shots finds the exact value before
//    every run the same way; each shot then searches the runs and walks one.
//
// Prediction only decides speed: every transfer is checked against the exact
// running value before it is used.
//
// A state of at most 14 qubits takes one launch for all of it.
#include <algorithm>
#include <climits>
#include <cmath>
#include <numeric>

#include "mh_internal.h"

namespace mh {
namespace {

constexpr uint32_t kBlockLog = 13;           // elements per block ...
constexpr uint32_t kSmallBlockLog = 11;      // ... and of a state of at most kSmallBlockQubits
constexpr uint32_t kSmallBlockQubits = 20;
constexpr uint32_t kGroup = 256;             // blocks per group
constexpr int kThreads = 256;
constexpr uint64_t kSat = uint64_t{1} << 62;  // saturation: "leaves the binade"
constexpr uint64_t kTop = (uint64_t{1} << 53) - 1;
constexpr int32_t kNonUniform = INT_MIN;

struct Xfer {
    uint64_t d0, d1;  // increment of K for input parity 0 / 1
    int32_t s;        // the binade's ulp exponent (kNonUniform: blocks disagree)
    uint32_t q;       // bit 0: output parity for input 0; bit 1: for input 1
};

__device__ __forceinline__ uint64_t sat_add(uint64_t a, uint64_t b) {
    const uint64_t c = a + b;
    return (c < a || c > kSat) ? kSat : c;
}

__device__ __forceinline__ Xfer identity_xfer(int32_t s) { return Xfer{0, 0, s, 0b10u}; }

// f then g.
__device__ __forceinline__ Xfer compose(const Xfer& f, const Xfer& g) {
    const uint32_t f0 = f.q & 1u, f1 = (f.q >> 1) & 1u;
    Xfer h;
    h.d0 = sat_add(f.d0, f0 ? g.d1 : g.d0);
    h.d1 = sat_add(f.d1, f1 ? g.d1 : g.d0);
    const uint32_t g0 = g.q & 1u, g1 = (g.q >> 1) & 1u;
    h.q = (f0 ? g1 : g0) | ((f1 ? g1 : g0) << 1);
    h.s = f.s == g.s ? f.s : kNonUniform;
    return h;
}

// The ulp exponent of the binade holding c >= 0.
__device__ __forceinline__ int32_t scale_of(double c) {
    const uint64_t bits = __double_as_longlong(c);
    const int32_t e = static_cast<int32_t>((bits >> 52) & 0x7FF);
    if (e <= 1) return -1074;  // subnormals and [2^-1022, 2^-1021) share ulp 2^-1074
    return e - 1075;
}

// c = K * 2^s exactly.
__device__ __forceinline__ uint64_t k_of(double c, int32_t s) {
    const uint64_t bits = __double_as_longlong(c);
    const uint64_t e = (bits >> 52) & 0x7FF;
    const uint64_t frac = bits & ((uint64_t{1} << 52) - 1);
    if (e == 0) return frac;                      // s == -1074
    const uint64_t m = frac | (uint64_t{1} << 52);
    return m << ((static_cast<int32_t>(e) - 1075) - s);  // 0 when normal binade; 1 for [2^-1022, 2^-1021)
}

__device__ __forceinline__ double value_of(uint64_t k, int32_t s) { return ldexp(static_cast<double>(k), s); }

// The step function of adding p at ulp 2^s.
__device__ __forceinline__ Xfer element_xfer(double p, int32_t s) {
    Xfer x = identity_xfer(s);
    if (p == 0.0) return x;
    const uint64_t bits = __double_as_longlong(p);
    const int32_t e = static_cast<int32_t>((bits >> 52) & 0x7FF);
    const uint64_t frac = bits & ((uint64_t{1} << 52) - 1);
    const uint64_t m = e == 0 ? frac : (frac | (uint64_t{1} << 52));
    const int32_t q = e == 0 ? -1074 : e - 1075;
    const int32_t shift = s - q;
    uint64_t r;
    bool tie = false;
    if (shift <= 0) {
        r = (-shift > 9) ? kSat : (m << (-shift));
    } else if (shift >= 64) {
        r = 0;
    } else {
        r = m >> shift;
        const uint64_t rem = m & ((uint64_t{1} << shift) - 1);
        const uint64_t half = uint64_t{1} << (shift - 1);
        if (rem > half) r += 1;
        tie = rem == half;
    }
    // Input parity P: d = r (+1 on a tie when P + r is odd); output parity (P + d) & 1.
    const uint64_t d0 = r + ((tie && (r & 1u)) ? 1u : 0u);
    const uint64_t d1 = r + ((tie && !(r & 1u)) ? 1u : 0u);
    x.d0 = d0;
    x.d1 = d1;
    x.q = static_cast<uint32_t>(d0 & 1u) | (static_cast<uint32_t>((1u + d1) & 1u) << 1);
    return x;
}

template <typename V>
__device__ __forceinline__ double prob(const V* s, uint64_t i) {
    const V v = s[i];
    const double x = static_cast<double>(v.x);
    const double y = static_cast<double>(v.y);
    return x * x + y * y;
}

struct SampleArgs {
    const void* state;
    uint64_t size;        // 2^n
    uint64_t block;       // elements per block
    uint32_t blocks;
    uint32_t groups;
    double* sums;         // [blocks]
    double* approx;       // [blocks] exclusive prefix of sums within the block's group
    double* gapprox;      // [groups] sum of a group, then the exclusive prefix of those from the carry
    Xfer* xfer;           // [blocks]
    Xfer* gxfer;          // [groups]
    double* cstart;       // [blocks + 1] exact c before each block
    uint32_t* jumped;     // [groups]
    // The exact running value before the first element (device; null: 0),
    // for a state that arrives in consecutive chunks.
    const double* carry;
    double unit;          // 1 / the whole state's bases: the guess for one element's probability
};

__device__ __forceinline__ double carry_of(const SampleArgs& a) { return a.carry ? *a.carry : 0.0; }

// v summed over the workgroup (a fixed order), in every thread.
__device__ __forceinline__ double block_sum(double v, double* waves) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = v + __shfl_xor(v, off, 64);
    __syncthreads();  // the sums of the call before are read
    if ((threadIdx.x & 63u) == 0) waves[threadIdx.x >> 6] = v;
    __syncthreads();
    v = waves[0];
#pragma unroll
    for (int w = 1; w < kThreads / 64; ++w) v = v + waves[w];
    return v;
}

// A block's transfer in the binade of ulp 2^s, where no element is a tie there:
// K grows by the same integer whatever its parity, the sum of the elements
// rounded to integers, in any order (the integers and their sums are exact in
// double below 2^53; a sum beyond leaves the binade, and stays beyond). Returns
// whether that holds; `sum` is the block's FP64 sum.
template <typename V>
__device__ __forceinline__ bool plain_xfer(const V* st, uint64_t i0, uint64_t count, int32_t s, double* waves,
                                           Xfer& x, double& sum) {
    double acc = 0.0, k = 0.0;
    bool tie = false;
#pragma unroll 8
    for (uint64_t i = threadIdx.x; i < count; i += kThreads) {
        const double p = prob(st, i0 + i);
        const double v = ldexp(p, -s), r = rint(v);
        acc = acc + p;
        k = k + r;
        tie = tie || fabs(v - r) == 0.5;
    }
    sum = block_sum(acc, waves);
    k = block_sum(k, waves);
    const bool any = __syncthreads_or(tie) != 0;
    const uint64_t d = k <= static_cast<double>(kTop) ? static_cast<uint64_t>(k) : kSat;
    const uint32_t odd = static_cast<uint32_t>(d & 1u);
    x = Xfer{d, d, s, odd | (odd ^ 1u) << 1};
    return !any;
}

// The only read of most of the state, and bound by it: 10,000 shots at 29
// qubits complex128 take 2.2 ms, 2.4 before the chain's steps in double, and 4.2
// with a read for the sums (1.4) and one for the transfers (1.9, bound by their
// integer steps as well as by the read). A
// block with a tie is left to block_xfer_kernel.
template <typename V>
__global__ void __launch_bounds__(kThreads) block_sums_kernel(SampleArgs a) {
    __shared__ double waves[kThreads / 64];
    const uint64_t b0 = uint64_t(blockIdx.x) * a.block;
    const double guess = carry_of(a) + (static_cast<double>(b0) + 0.5 * static_cast<double>(a.block)) * a.unit;
    Xfer x;
    double sum;
    const bool plain = plain_xfer(static_cast<const V*>(a.state), b0, a.block, scale_of(guess), waves, x, sum);
    if (!plain) x.s = kNonUniform;
    if (threadIdx.x == 0) {
        a.sums[blockIdx.x] = sum;
        a.xfer[blockIdx.x] = x;
    }
}

// The inclusive sum over a workgroup's threads (any order: predictions only).
template <uint32_t kWaves>
__device__ __forceinline__ double inclusive_sum(double v, double* waves) {
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const double u = __shfl_up(v, off, 64);
        if (lane >= static_cast<uint32_t>(off)) v = v + u;
    }
    if (lane == 63) waves[wave] = v;
    __syncthreads();
    for (uint32_t w = 0; w < wave; ++w) v = v + waves[w];
    return v;
}

// A workgroup per group: the exclusive prefix of its block sums and its total
// (for a single group, the carry in its place).
__global__ void __launch_bounds__(kThreads) group_prefix_kernel(SampleArgs a) {
    __shared__ double waves[kThreads / 64];
    const uint32_t b = blockIdx.x * kGroup + threadIdx.x;
    const double v = b < a.blocks ? a.sums[b] : 0.0;
    const double inc = inclusive_sum<kThreads / 64>(v, waves);
    if (b < a.blocks) a.approx[b] = inc - v;
    if (threadIdx.x == kThreads - 1) a.gapprox[blockIdx.x] = a.groups == 1 ? carry_of(a) : inc;
}

// One workgroup: the groups' totals become the sums before each group.
__global__ void __launch_bounds__(1024) approx_prefix_kernel(SampleArgs a) {
    __shared__ double waves[1024 / 64];
    double run = carry_of(a);
    for (uint32_t g0 = 0; g0 < a.groups; g0 += 1024) {
        const uint32_t g = g0 + threadIdx.x;
        const double v = g < a.groups ? a.gapprox[g] : 0.0;
        const double inc = inclusive_sum<1024 / 64>(v, waves);
        if (g < a.groups) a.gapprox[g] = run + (inc - v);
        double total = 0.0;
        for (uint32_t w = 0; w < 1024 / 64; ++w) total = w == 0 ? waves[0] : total + waves[w];
        run = run + total;
        __syncthreads();  // the wave sums are read before the next round writes them
    }
}

// Amplitudes of a block staged in LDS at a time by block_xfer_kernel: 16 KiB,
// so that several workgroups share a CU (a whole block of 2^13, 64 KiB, left
// room for two and the kernel latency-bound).
constexpr uint32_t kXferStage = 2048;

// The blocks whose transfer was not found in the predicted binade: again
// without order where they have no tie, else run by run.
template <typename V>
__global__ void __launch_bounds__(kThreads) block_xfer_kernel(SampleArgs a) {
    __shared__ double p_sh[kXferStage];
    __shared__ Xfer red[kThreads];
    const V* st = static_cast<const V*>(a.state);
    const uint32_t b = blockIdx.x;
    const int32_t s = scale_of(a.gapprox[b / kGroup] + a.approx[b]);
    const uint64_t i0 = uint64_t(b) * a.block;
    const int32_t found = a.xfer[b].s;
    if (found == s) return;
    if (found != kNonUniform) {
        Xfer x;
        double sum;
        if (plain_xfer(st, i0, a.block, s, p_sh, x, sum)) {
            if (threadIdx.x == 0) a.xfer[b] = x;
            return;
        }
        __syncthreads();  // the sums in p_sh are read
    }
    const uint32_t stage = static_cast<uint32_t>(min(a.block, uint64_t{kXferStage}));
    Xfer total = identity_xfer(s);  // thread 0's: the stages composed in order
    for (uint64_t base = 0; base < a.block; base += stage) {
        for (uint32_t i = threadIdx.x; i < stage; i += kThreads) p_sh[i] = prob(st, i0 + base + i);
        __syncthreads();
        // Each thread composes a contiguous run in order; then a fixed tree
        // (the composition is exact, so the order only has to respect the
        // sequence). The tree's barriers also end every read of p_sh and red
        // before the next stage writes them.
        const uint32_t per = (stage + kThreads - 1) / kThreads;
        const uint32_t j0 = min(stage, threadIdx.x * per);
        const uint32_t j1 = min(stage, j0 + per);
        Xfer acc = identity_xfer(s);
        for (uint32_t j = j0; j < j1; ++j) acc = compose(acc, element_xfer(p_sh[j], s));
        red[threadIdx.x] = acc;
        __syncthreads();
        for (int stride = 1; stride < kThreads; stride <<= 1) {
            if ((threadIdx.x % (2 * stride)) == 0) red[threadIdx.x] = compose(red[threadIdx.x], red[threadIdx.x + stride]);
            __syncthreads();
        }
        if (threadIdx.x == 0) total = compose(total, red[0]);
    }
    if (threadIdx.x == 0) a.xfer[b] = total;
}

__global__ void __launch_bounds__(kThreads) group_xfer_kernel(SampleArgs a) {
    __shared__ Xfer red[kThreads];
    const uint32_t g = blockIdx.x;
    const uint32_t b = g * kGroup + threadIdx.x;
    red[threadIdx.x] = b < a.blocks ? a.xfer[b] : identity_xfer(a.xfer[g * kGroup].s);
    __syncthreads();
    for (int stride = 1; stride < kThreads; stride <<= 1) {
        if ((threadIdx.x % (2 * stride)) == 0) red[threadIdx.x] = compose(red[threadIdx.x], red[threadIdx.x + stride]);
        __syncthreads();
    }
    if (threadIdx.x == 0) a.gxfer[g] = red[0];
}

// ---- scans of transfers over a workgroup

// A transfer of one binade (the scan's own: all of them share it).
struct Step {
    uint64_t d0, d1;
    uint32_t q;
};

__device__ __forceinline__ Step then(const Step& f, const Step& g) {
    const uint32_t f0 = f.q & 1u, f1 = (f.q >> 1) & 1u;
    Step h;
    h.d0 = sat_add(f.d0, f0 ? g.d1 : g.d0);
    h.d1 = sat_add(f.d1, f1 ? g.d1 : g.d0);
    h.q = ((g.q >> f0) & 1u) | (((g.q >> f1) & 1u) << 1);
    return h;
}

__device__ __forceinline__ Step shift_up(const Step& x, int by) {
    Step r;
    r.d0 = static_cast<uint64_t>(__shfl_up(static_cast<unsigned long long>(x.d0), by, 64));
    r.d1 = static_cast<uint64_t>(__shfl_up(static_cast<unsigned long long>(x.d1), by, 64));
    r.q = static_cast<uint32_t>(__shfl_up(static_cast<int>(x.q), by, 64));
    return r;
}

struct ScanShared {
    Step wave[kThreads / 64];
    uint32_t bad[kThreads / 64];
};

// Where a chain that starts from c at thread `from` gets to: thread t's start
// and end values (exact for from <= t < the returned index, and its start for
// that index itself), each thread applying `x` (`ok`: it is of c's binade and
// may be used). Returns the first thread whose transfer does not apply, or
// kThreads. Every thread of the workgroup calls it.
__device__ __forceinline__ uint32_t follow(ScanShared& sh, double c, int32_t s, Step x, bool ok, uint32_t from,
                                           double& start, double& end) {
    const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
    const Step none{0, 0, 0b10u};
    Step inc = t >= from ? x : none;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const Step f = shift_up(inc, off);
        if (lane >= static_cast<uint32_t>(off)) inc = then(f, inc);
    }
    Step exc = shift_up(inc, 1);
    if (lane == 0) exc = none;
    if (lane == 63) sh.wave[wave] = inc;
    __syncthreads();
    Step pre = none;
    for (uint32_t w = 0; w < wave; ++w) pre = then(pre, sh.wave[w]);
    inc = then(pre, inc);
    exc = then(pre, exc);
    const uint64_t k = k_of(c, s);
    const uint64_t k0 = sat_add(k, (k & 1u) ? exc.d1 : exc.d0);
    const uint64_t k1 = sat_add(k, (k & 1u) ? inc.d1 : inc.d0);
    start = value_of(k0, s);
    end = value_of(k1, s);
    const uint64_t bad = __ballot(t >= from && (!ok || k1 > kTop));
    if (lane == 0) sh.bad[wave] = bad ? wave * 64 + static_cast<uint32_t>(__ffsll(static_cast<unsigned long long>(bad))) - 1 : kThreads;
    __syncthreads();
    uint32_t first = kThreads;
#pragma unroll
    for (uint32_t w = 0; w < kThreads / 64; ++w) first = min(first, sh.bad[w]);
    return first;
}

// Elements exact_stage takes at a time: eight to a thread, 16 KiB of LDS.
constexpr uint32_t kStage = 2048;

struct StageShared {
    ScanShared scan;
    double p[kStage];
    double start[kThreads + 1];  // the exact running value before each run; the last: after the stage
    double c;
};

// The step of the elements p[j0..j1) at ulp 2^s, in double: each element's
// nearest integer (a tie's even one, or its odd one where K is odd there), and
// for both parities of K the sum and where it leads. The sums are exact below
// 2^53; beyond they leave the binade, and stay beyond.
__device__ __forceinline__ Step run_step(const double* p, uint32_t j0, uint32_t j1, int32_t s) {
    double k0 = 0.0, k1 = 0.0;
    bool q0 = false, q1 = true;  // K's parity after the elements so far, for an even and an odd start
#pragma unroll 2
    for (uint32_t j = j0; j < j1; ++j) {
        const double v = ldexp(p[j], -s), r = rint(v), off = v - r;
        const bool tie = fabs(off) == 0.5;
        const double h = r * 0.5;
        const bool odd = rint(h) != h;
        const double up = r + (off + off);  // a tie's odd neighbour
        k0 = k0 + (tie && q0 ? up : r);
        k1 = k1 + (tie && q1 ? up : r);
        q0 = !tie && (q0 != odd);
        q1 = !tie && (q1 != odd);
    }
    constexpr double top = static_cast<double>(kTop);
    return Step{k0 <= top ? static_cast<uint64_t>(k0) : kSat, k1 <= top ? static_cast<uint64_t>(k1) : kSat,
                static_cast<uint32_t>(q0) | static_cast<uint32_t>(q1) << 1};
}

// Runs that one thread walks where the running value leaves its binade: near
// the start of a state the next binade ends soon after (calls with 1, 2, 4 runs:
// 10 qubits 56, 52, 54 us, 17 qubits 232, 223, 216, a layered state of 24 1226,
// 1239, 1250; 16 and more only lose).
constexpr uint32_t kWalk = 2;

// The stage's probabilities in sh.p (count of them) from the exact running
// value c: every run's start into sh.start, the value after them into
// sh.start[kThreads]. A run is `per` consecutive elements. Each round ends at
// the first run that leaves the binade, from which one thread walks kWalk.
__device__ __forceinline__ void exact_stage(StageShared& sh, uint32_t count, double c) {
    const uint32_t t = threadIdx.x, per = (count + kThreads - 1) / kThreads;
    const uint32_t j0 = min(count, t * per), j1 = min(count, j0 + per);
    uint32_t from = 0;
    while (true) {
        if (c != c) {  // a NaN stays one (it has no binade: its steps would say otherwise)
            if (t >= from) sh.start[t] = c;
            if (t == 0) sh.start[kThreads] = c;
            break;
        }
        const int32_t s = scale_of(c);
        Step x{0, 0, 0b10u};
        if (t >= from) x = run_step(sh.p, j0, j1, s);
        double start, end;
        const uint32_t first = follow(sh.scan, c, s, x, true, from, start, end);
        if (t >= from && t <= first) sh.start[t] = start;
        if (first == kThreads) {
            if (t == kThreads - 1) sh.start[kThreads] = end;
            break;
        }
        from = min(first + kWalk, static_cast<uint32_t>(kThreads));
        if (t == first) {
            for (uint32_t r = first; r < from; ++r) {
                sh.start[r] = start;
                const uint32_t e = min(count, (r + 1) * per);
#pragma unroll 8
                for (uint32_t j = min(count, r * per); j < e; ++j) start = start + sh.p[j];
            }
            sh.c = start;
            if (from == kThreads) sh.start[kThreads] = start;
        }
        __syncthreads();
        if (from == kThreads) break;
        c = sh.c;
    }
    __syncthreads();
}

// The probabilities of `count` elements from index i0 into sh.p; every thread
// is past its reads of the stage before.
template <typename V>
__device__ __forceinline__ void load_stage(StageShared& sh, const V* st, uint64_t i0, uint32_t count) {
    for (uint32_t i = threadIdx.x; i < count; i += kThreads) sh.p[i] = prob(st, i0 + i);
    __syncthreads();
}

// One workgroup: the exact chain over all blocks, bound by its own latency (a
// scan of 256 transfers takes about 2 us, and each binade crossing three of
// them and a walk). 29 qubits: 0.52 ms, 17 qubits 0.11 (0.75 and 0.14 with the
// elements' steps in integers); one thread applying the transfers and 32
// composing a dirty block's sub-blocks took 3.77 and 1.35.
template <typename V>
__global__ void __launch_bounds__(kThreads) chain_kernel(SampleArgs a) {
    __shared__ StageShared sh;
    const V* st = static_cast<const V*>(a.state);
    const uint32_t t = threadIdx.x;
    const uint32_t stage = static_cast<uint32_t>(min(a.block, uint64_t{kStage}));
    double c = carry_of(a);
    if (t == 0) a.cstart[0] = c;
    // Once the sum is NaN (after block b - 1, in group g) it stays NaN.
    auto rest = [&](uint32_t g, uint32_t b) {
        for (uint64_t i = uint64_t(b) + t; i <= a.blocks; i += kThreads) a.cstart[i] = c;
        for (uint32_t i = g + t; i < a.groups; i += kThreads) a.jumped[i] = 0;
    };
    if (c != c) return rest(0, 0);
    for (uint32_t g = 0; g < a.groups;) {
        // Whole groups while they apply.
        {
            const uint32_t count = min(static_cast<uint32_t>(kThreads), a.groups - g);
            const int32_t s = scale_of(c);
            Xfer x = identity_xfer(s);
            if (t < count) x = a.gxfer[g + t];
            double start, end;
            const uint32_t first = min(count, follow(sh.scan, c, s, Step{x.d0, x.d1, x.q}, x.s == s, 0, start, end));
            if (t < first) {
                a.jumped[g + t] = 1;
                a.cstart[min(a.blocks, (g + t + 1) * kGroup)] = end;
            }
            if (t == first) sh.c = start;
            if (first == kThreads && t == kThreads - 1) sh.c = end;
            __syncthreads();
            c = sh.c;
            __syncthreads();
            g += first;
            if (first == count) continue;
        }
        // Group g block by block, and its blocks that do not apply element by
        // element.
        if (t == 0) a.jumped[g] = 0;
        const uint32_t end_block = min(a.blocks, (g + 1) * kGroup);
        for (uint32_t b = g * kGroup; b < end_block;) {
            const uint32_t count = end_block - b;
            const int32_t s = scale_of(c);
            Xfer x = identity_xfer(s);
            if (t < count) x = a.xfer[b + t];
            double start, end;
            const uint32_t first = min(count, follow(sh.scan, c, s, Step{x.d0, x.d1, x.q}, x.s == s, 0, start, end));
            if (t < first) a.cstart[b + t + 1] = end;
            if (t == first) sh.c = start;
            if (first == kThreads && t == kThreads - 1) sh.c = end;
            __syncthreads();
            c = sh.c;
            __syncthreads();
            b += first;
            if (first == count) continue;
            for (uint64_t at = 0; at < a.block; at += stage) {
                load_stage(sh, st, uint64_t(b) * a.block + at, stage);
                exact_stage(sh, stage, c);
                c = sh.start[kThreads];
                __syncthreads();
            }
            ++b;
            if (c != c) return rest(g, b);
            if (t == 0) a.cstart[b] = c;
        }
        ++g;
    }
}

// Block starts inside the groups the chain jumped over.
__global__ void __launch_bounds__(kThreads) expand_kernel(SampleArgs a) {
    __shared__ ScanShared sh;
    const uint32_t g = blockIdx.x, t = threadIdx.x;
    if (!a.jumped[g]) return;
    const uint32_t b0 = g * kGroup;
    const uint32_t count = min(kGroup, a.blocks - b0);
    const double c = a.cstart[b0];
    const int32_t s = scale_of(c);
    Xfer x = identity_xfer(s);
    if (t < count) x = a.xfer[b0 + t];
    double start, end;
    follow(sh, c, s, Step{x.d0, x.d1, x.q}, true, 0, start, end);  // valid: the whole group was
    if (t + 1 < count) a.cstart[b0 + t + 1] = end;
}

// The first index of the stage at i0 whose running sum exceeds x, or `none`
// (the sum turned NaN first: from there on it exceeds nothing), for an x that
// the stage's end is not at most: its run by bisection, then plain adds from
// the run's exact start.
__device__ __forceinline__ uint64_t resolve(const StageShared& sh, uint32_t count, uint64_t i0, double x,
                                            uint64_t none) {
    uint32_t lo = 0, hi = kThreads - 1;  // the first run r whose end start[r + 1] is not at most x
    while (lo < hi) {
        const uint32_t mid = (lo + hi) / 2;
        if (!(x >= sh.start[mid + 1]))
            hi = mid;
        else
            lo = mid + 1;
    }
    const uint32_t per = (count + kThreads - 1) / kThreads;
    const uint32_t j0 = min(count, lo * per), j1 = min(count, j0 + per);
    double c = sh.start[lo];
    for (uint32_t j = j0; j < j1; ++j) {
        c = c + sh.p[j];
        if (x < c) return i0 + j;
    }
    return none;
}

// Shots a workgroup takes from one reading of their block, at most.
constexpr uint32_t kShare = 1024;

// Workgroup i has shots [i * piece, (i + 1) * piece), piece a divisor of kShare
// (1 unless they are sorted and all of the state's). Sorted uniforms: the first
// shot of a block, and each whose number is a multiple of kShare, takes the
// shots of its block up to the next such; the others leave theirs to it. Else
// each takes its own. Every uniform gets the first index whose running sum exceeds it (one
// below 0 index 0), else the last index; for one chunk of a state (`partial`, `first_index` the chunk's first index) one
// that another chunk's sums exceed first is left alone. Comparisons are with
// "at most", so that the searches hold where the sum turns NaN, which exceeds
// nothing.
//
// A block's elements are read once for all of its shots, all of them in
// parallel: 0.22 ms for 10,000 shots at 29 qubits (1.3 GB of blocks), 0.045 for
// 4096 at 17; walking them with one thread per shot took 2.26 and 1.24.
template <typename V>
__global__ void __launch_bounds__(kThreads) shots_kernel(SampleArgs a, const double* u, uint64_t shots, uint64_t* out,
                                                        uint64_t first_index, bool sorted, bool partial,
                                                        uint32_t piece) {
    __shared__ StageShared sh;
    const uint32_t t = threadIdx.x;
    const uint64_t begin = uint64_t(blockIdx.x) * piece, end = min(begin + piece, shots);
    const bool opens = first_index == 0;  // nothing comes before this state (or chunk)
    for (uint64_t i = begin; i < end;) {
        const double x = u[i];
        if (partial && (x >= a.cstart[a.blocks] || !(opens || x >= a.cstart[0]))) return;
        // The first block whose end value is not at most x, kThreads pivots at a
        // time.
        uint32_t lo = 0, hi = a.blocks;  // the answer is in [lo, hi]
        while (lo < hi) {
            const uint32_t step = (hi - lo + kThreads - 1) / kThreads;
            const uint64_t at = uint64_t(lo) + uint64_t(t + 1) * step - 1;  // the last block of the thread's share
            const bool past = at < hi && x >= a.cstart[at + 1];
            const uint32_t shares = static_cast<uint32_t>(__syncthreads_count(past));
            const uint64_t from = uint64_t(lo) + uint64_t(shares) * step;
            const uint32_t limit = hi;
            lo = static_cast<uint32_t>(min(from, uint64_t{limit}));
            hi = static_cast<uint32_t>(min(from + step - 1, uint64_t{limit}));
        }
        if (lo == a.blocks) {  // sorted: the later ones as well
            for (uint64_t j = i + t; j < end; j += kThreads) out[j] = first_index + a.size - 1;
            return;
        }
        const double c0 = a.cstart[lo], c1 = a.cstart[lo + 1];
        const bool takes = !sorted || i % kShare == 0 || !((opens && lo == 0) || u[i - 1] >= c0);
        uint64_t count = 1;
        if (sorted) {
            const uint64_t limit = takes ? min(shots, (i / kShare + 1) * kShare) : end;
            count = 0;
            for (uint32_t more = kThreads; more == kThreads;) {
                const uint64_t at = i + count + t;
                more = static_cast<uint32_t>(__syncthreads_count(at < limit && !(u[at] >= c1)));
                count += more;
            }
        }
        if (takes) {
            const double last = u[i + count - 1];
            const V* st = static_cast<const V*>(a.state);
            const uint32_t stage = static_cast<uint32_t>(min(a.block, uint64_t{kStage}));
            double c = c0;
            for (uint64_t at = 0; at < a.block; at += stage) {
                const uint64_t i0 = uint64_t(lo) * a.block + at;
                load_stage(sh, st, i0, stage);
                exact_stage(sh, stage, c);
                c = sh.start[kThreads];
                for (uint64_t j = t; j < count; j += kThreads) {
                    const double y = u[i + j];
                    // A NaN: an earlier stage's sums, if any, were at most y.
                    if ((at == 0 || y >= sh.start[0]) && !(y >= c)) {
                        const uint64_t hit = resolve(sh, stage, i0, y, UINT64_MAX);
                        if (hit != UINT64_MAX)
                            out[i + j] = first_index + hit;
                        else if (!partial)
                            out[i + j] = a.size - 1;
                    }
                }
                __syncthreads();
                if (!(last >= c)) break;
            }
        }
        i += count;
    }
}

// A thread per shot, in any order: its block by bisection, then plain adds from
// the block's start (bound by their latency, so for many shots only).
template <typename V>
__global__ void __launch_bounds__(kThreads) shots_walk_kernel(SampleArgs a, const double* u, uint64_t shots,
                                                             uint64_t* out) {
    const uint64_t t = uint64_t(blockIdx.x) * kThreads + threadIdx.x;
    if (t >= shots) return;
    const double x = u[t];
    uint32_t lo = 0, hi = a.blocks;  // the first block whose end value is not at most x
    while (lo < hi) {
        const uint32_t mid = (lo + hi) / 2;
        if (!(x >= a.cstart[mid + 1]))
            hi = mid;
        else
            lo = mid + 1;
    }
    uint64_t hit = a.size - 1;
    if (lo < a.blocks) {
        const V* st = static_cast<const V*>(a.state);
        const uint64_t i0 = uint64_t(lo) * a.block;
        double c = a.cstart[lo];
        for (uint64_t i = 0; i < a.block; ++i) {
            c = c + prob(st, i0 + i);
            if (x < c) {
                hit = i0 + i;
                break;
            }
        }
    }
    out[t] = hit;
}

// A small state's shots (any order), kShare of them a workgroup, each stage by
// stage.
template <typename V>
__global__ void __launch_bounds__(kThreads) small_shots_kernel(const V* st, uint32_t size, const double* u,
                                                              uint64_t shots, uint64_t* out) {
    __shared__ StageShared sh;
    const uint64_t begin = uint64_t(blockIdx.x) * kShare, last = min(begin + kShare, shots);
    double c = 0.0;
    for (uint32_t i0 = 0; i0 < size; i0 += kStage) {
        const uint32_t count = min(size - i0, kStage);
        load_stage(sh, st, i0, count);
        exact_stage(sh, count, c);
        const bool end = i0 + count == size;
        c = sh.start[kThreads];
        for (uint64_t j = begin + threadIdx.x; j < last; j += kThreads) {
            const double y = u[j];
            if ((i0 == 0 || y >= sh.start[0]) && !(y >= c))
                out[j] = resolve(sh, count, i0, y, size - 1);
            else if (end && y >= c)
                out[j] = size - 1;
        }
        __syncthreads();
    }
}

__global__ void __launch_bounds__(kThreads) fill_index_kernel(uint64_t* out, uint64_t count, uint64_t value) {
    const uint64_t t = uint64_t(blockIdx.x) * kThreads + threadIdx.x;
    if (t < count) out[t] = value;
}

// The first half of the sampler over one state: the exact running value at
// every block start (block sums, predicted binades, composed transfers, the
// chain, the starts inside jumped groups), in device tables kept for draws.
struct SamplerTables {
    DeviceBuffer buf;
    SampleArgs a{};
};

uint64_t r16(uint64_t bytes) { return (bytes + 15) / 16 * 16; }

uint64_t block_of(uint32_t n) {
    return uint64_t{1} << std::min<uint32_t>(n, n <= kSmallBlockQubits ? kSmallBlockLog : kBlockLog);
}

uint64_t table_bytes(uint32_t n) {
    const uint64_t nb = (uint64_t{1} << n) / block_of(n), groups = (nb + kGroup - 1) / kGroup;
    return r16(nb * sizeof(Xfer)) + r16(groups * sizeof(Xfer)) + r16(nb * sizeof(double)) +
           2 * r16((nb + 1) * sizeof(double)) + r16(groups * sizeof(double)) + r16(groups * sizeof(uint32_t));
}

// Allocates the tables of a state of 2^n amplitudes at `state`, or of such a
// chunk of a state of `whole` qubits.
void layout_tables(SamplerTables& t, const void* state, uint32_t n, uint32_t whole) {
    context();
    SampleArgs& a = t.a;
    a.state = state;
    a.size = uint64_t{1} << n;
    a.block = block_of(n);
    a.blocks = static_cast<uint32_t>(a.size / a.block);
    a.groups = (a.blocks + kGroup - 1) / kGroup;
    const uint64_t nb = a.blocks;
    t.buf = DeviceBuffer(table_bytes(n));
    char* p = t.buf.as<char>();
    auto take = [&](uint64_t bytes) {
        char* r = p;
        p += r16(bytes);
        return r;
    };
    a.xfer = reinterpret_cast<Xfer*>(take(nb * sizeof(Xfer)));
    a.gxfer = reinterpret_cast<Xfer*>(take(uint64_t(a.groups) * sizeof(Xfer)));
    a.sums = reinterpret_cast<double*>(take(nb * sizeof(double)));
    a.approx = reinterpret_cast<double*>(take((nb + 1) * sizeof(double)));
    a.cstart = reinterpret_cast<double*>(take((nb + 1) * sizeof(double)));
    a.gapprox = reinterpret_cast<double*>(take(uint64_t(a.groups) * sizeof(double)));
    a.jumped = reinterpret_cast<uint32_t*>(take(uint64_t(a.groups) * sizeof(uint32_t)));
    a.carry = nullptr;
    a.unit = std::ldexp(1.0, -static_cast<int>(whole));
}

// Queues the table kernels for the state and carry in `a` on `stream`.
template <typename V>
void launch_tables(const SampleArgs& a, hipStream_t stream) {
    hipLaunchKernelGGL(block_sums_kernel<V>, dim3(a.blocks), dim3(kThreads), 0, stream, a);
    MH_HIP(hipGetLastError());
    hipLaunchKernelGGL(group_prefix_kernel, dim3(a.groups), dim3(kThreads), 0, stream, a);
    MH_HIP(hipGetLastError());
    if (a.groups > 1) {
        hipLaunchKernelGGL(approx_prefix_kernel, dim3(1), dim3(1024), 0, stream, a);
        MH_HIP(hipGetLastError());
    }
    hipLaunchKernelGGL(block_xfer_kernel<V>, dim3(a.blocks), dim3(kThreads), 0, stream, a);
    MH_HIP(hipGetLastError());
    hipLaunchKernelGGL(group_xfer_kernel, dim3(a.groups), dim3(kThreads), 0, stream, a);
    MH_HIP(hipGetLastError());
    hipLaunchKernelGGL(chain_kernel<V>, dim3(1), dim3(kThreads), 0, stream, a);
    MH_HIP(hipGetLastError());
    hipLaunchKernelGGL(expand_kernel, dim3(a.groups), dim3(kThreads), 0, stream, a);
    MH_HIP(hipGetLastError());
}

template <typename V>
void prepare_tables(SamplerTables& t, const void* state, uint32_t n) {
    layout_tables(t, state, n, n);
    launch_tables<V>(t.a, streams().main);
}

// States sampled without tables, in one launch: eight stages. Whole calls, this
// form against the tables': 10 qubits and 100 shots 54 against 124 us, 14 qubits
// and 1000 shots 110 against 175, 15 qubits 174 against 176. All of a state's
// shots by one workgroup took 14.4 ms for 2,000,000 at 10 qubits, kShare a
// workgroup 2.3.
constexpr uint32_t kSmallQubits = 14;

// Draws from a kept state of that size take this form too if it is one stage or
// there are many of them (12 qubits, 1000 and 10,000 draws: 78 and 90 us, 78 and
// 283 from the tables; 14 qubits 147 and 168, 73 and 184).
constexpr uint64_t kSmallDraws = 4096;

// Sorted shots go to about this many workgroups or more, up to kMostPiece of
// them each (2,000,000 shots of 17 and 27 qubits, ms: 4096 workgroups 2.6 and
// 6.9, 16384 2.9 and 5.3, 65536 3.4 and 6.3, one a shot 4.4 and 7.5).
constexpr uint64_t kPieces = 16384;
constexpr uint32_t kMostPiece = 256;
static_assert(kShare % kMostPiece == 0);

// Of so many shots in no order each walks its block by itself where the state
// stays in the caches: a workgroup a shot reads the block for that one alone
// (10,000, 100,000 and 2,000,000 draws: 16 qubits 0.33, 0.46 and 5.9 ms walked,
// 0.15, 0.94 and 17 so; 21 qubits, with longer blocks, 1.4, 1.6 and 17, 0.24, 1.7
// and 32; 23 qubits 1.6, 2.1 and 39, 0.21, 1.6 and 30).
constexpr uint32_t kWalkQubits = 22;
bool walked(const SampleArgs& a, uint64_t shots) {
    return a.size <= (uint64_t{1} << kWalkQubits) && shots > (a.size <= (uint64_t{1} << kSmallBlockQubits) ? 1u << 15 : 1u << 16);
}

// A launch takes fewer than 2^32 threads.
constexpr uint64_t kMaxGrid = uint64_t{1} << 23;
static_assert(kMaxGrid * kThreads < uint64_t{1} << 32);

// Queues the shots of a state (or chunk) whose tables are ready.
template <typename V>
void launch_shots(const SampleArgs& a, const double* u, uint64_t shots, uint64_t* out, uint64_t first_index,
                  bool sorted, bool partial, hipStream_t stream) {
    uint32_t piece = 1;
    if (sorted && !partial)
        while (piece < kMostPiece && shots / (2 * piece) >= kPieces) piece *= 2;
    for (uint64_t at = 0; at < shots; at += kMaxGrid * piece) {
        const uint64_t count = std::min(shots - at, kMaxGrid * piece);
        hipLaunchKernelGGL(shots_kernel<V>, dim3(static_cast<uint32_t>((count + piece - 1) / piece)), dim3(kThreads), 0,
                           stream, a, u + at, count, out + at, first_index, sorted, partial, piece);
        MH_HIP(hipGetLastError());
    }
}

template <typename V>
void launch_walks(const SampleArgs& a, const double* u, uint64_t shots, uint64_t* out, hipStream_t stream) {
    for (uint64_t at = 0; at < shots; at += kMaxGrid * kThreads) {
        const uint64_t count = std::min(shots - at, kMaxGrid * kThreads);
        hipLaunchKernelGGL(shots_walk_kernel<V>, dim3(static_cast<uint32_t>((count + kThreads - 1) / kThreads)),
                           dim3(kThreads), 0, stream, a, u + at, count, out + at);
        MH_HIP(hipGetLastError());
    }
}

template <typename V>
void launch_small_shots(const V* state, uint32_t size, const double* u, uint64_t shots, uint64_t* out,
                        hipStream_t stream) {
    for (uint64_t at = 0; at < shots; at += kMaxGrid * kShare) {
        const uint64_t count = std::min(shots - at, kMaxGrid * kShare);
        hipLaunchKernelGGL(small_shots_kernel<V>, dim3(static_cast<uint32_t>((count + kShare - 1) / kShare)),
                           dim3(kThreads), 0, stream, state, size, u + at, count, out + at);
        MH_HIP(hipGetLastError());
    }
}

// Device copies of a call's uniforms, and its indices.
struct ShotBuffers {
    DeviceBuffer io;
    double* u = nullptr;
    uint64_t* out = nullptr;
    ShotBuffers(const double* uniforms, uint64_t count) : io(2 * r16(count * sizeof(double))) {
        u = io.as<double>();
        out = reinterpret_cast<uint64_t*>(io.as<char>() + r16(count * sizeof(double)));
        upload(u, uniforms, count * sizeof(double));
    }
};

// The second half: each uniform's basis index (any order), waited for.
template <typename V>
void draw_basis(const SampleArgs& a, const double* uniforms, uint64_t count, uint64_t* basis_out) {
    if (count == 0) return;
    context();
    ShotBuffers shots(uniforms, count);
    const bool sorted = std::is_sorted(uniforms, uniforms + count);
    if (a.size <= kStage || (a.size <= (uint64_t{1} << kSmallQubits) && count >= kSmallDraws))
        launch_small_shots(static_cast<const V*>(a.state), static_cast<uint32_t>(a.size), shots.u, count, shots.out,
                           streams().main);
    else if (!sorted && walked(a, count))
        launch_walks<V>(a, shots.u, count, shots.out, streams().main);
    else
        launch_shots<V>(a, shots.u, count, shots.out, 0, sorted, false, streams().main);
    download(basis_out, shots.out, count * sizeof(uint64_t));
}

template <typename V>
void run_sampler(const void* state, uint32_t n, const double* sorted_u, uint64_t shots, uint64_t* basis_out) {
    if (n <= kSmallQubits) {
        context();
        ShotBuffers io(sorted_u, shots);
        launch_small_shots(static_cast<const V*>(state), 1u << n, io.u, shots, io.out, streams().main);
        download(basis_out, io.out, shots * sizeof(uint64_t));
        return;
    }
    SamplerTables t;
    prepare_tables<V>(t, state, n);
    draw_basis<V>(t.a, sorted_u, shots, basis_out);
}

}  // namespace

void sample_sorted(const void* state, uint32_t n, int32_t precision, const double* sorted_u, uint64_t shots,
                   uint64_t* basis_out) {
    amp_bytes(precision);
    if (n > 40) fail(MH_ERR_INVALID, "sample: num_qubits above 40");
    if (shots == 0) return;
    for (uint64_t i = 1; i < shots; ++i)
        if (!(sorted_u[i - 1] <= sorted_u[i])) fail(MH_ERR_INVALID, "sample: uniforms are not sorted");
    if (precision == MH_C128)
        run_sampler<double2>(state, n, sorted_u, shots, basis_out);
    else
        run_sampler<float2>(state, n, sorted_u, shots, basis_out);
}

uint32_t sampler_launches(uint32_t n) {
    if (n <= kSmallQubits) return 1;
    return (uint64_t{1} << n) / block_of(n) > kGroup ? 8 : 7;
}

uint64_t sampler_table_bytes(uint32_t n) { return n <= kSmallQubits ? 0 : table_bytes(n); }

struct ChunkedSampler::Impl {
    uint32_t n = 0, chunk_log = 0;
    int32_t precision = MH_C128;
    uint64_t shots = 0, next = 0;
    hipStream_t stream = nullptr;
    SamplerTables tables[2];
    DeviceBuffer io;  // uniforms, basis indices, the zero carry of chunk 0
    double* du = nullptr;
    uint64_t* dout = nullptr;
    double* zero = nullptr;
};

ChunkedSampler::ChunkedSampler(uint32_t n, uint32_t chunk_log, int32_t precision, const double* sorted_u,
                               uint64_t shots, hipStream_t stream)
    : impl_(std::make_unique<Impl>()) {
    amp_bytes(precision);
    if (n > 40 || chunk_log > n) fail(MH_ERR_INVALID, "chunked sampler: chunk above the state or above 40 qubits");
    for (uint64_t i = 1; i < shots; ++i)
        if (!(sorted_u[i - 1] <= sorted_u[i])) fail(MH_ERR_INVALID, "sample: uniforms are not sorted");
    Impl& m = *impl_;
    m.n = n;
    m.chunk_log = chunk_log;
    m.precision = precision;
    m.shots = shots;
    m.stream = stream;
    for (SamplerTables& t : m.tables) layout_tables(t, nullptr, chunk_log, n);
    m.io = DeviceBuffer(r16(std::max<uint64_t>(shots, 1) * sizeof(double)) +
                        r16(std::max<uint64_t>(shots, 1) * sizeof(uint64_t)) + 16);
    m.du = m.io.as<double>();
    m.dout = reinterpret_cast<uint64_t*>(m.io.as<char>() + r16(std::max<uint64_t>(shots, 1) * sizeof(double)));
    m.zero = reinterpret_cast<double*>(reinterpret_cast<char*>(m.dout) + r16(std::max<uint64_t>(shots, 1) * sizeof(uint64_t)));
    MH_HIP(hipMemsetAsync(m.zero, 0, sizeof(double), stream));
    if (shots > 0) {
        MH_HIP(hipMemcpyAsync(m.du, sorted_u, shots * sizeof(double), hipMemcpyHostToDevice, stream));
        // A uniform at or above the total goes to the last index.
        hipLaunchKernelGGL(fill_index_kernel, dim3(static_cast<uint32_t>((shots + kThreads - 1) / kThreads)),
                           dim3(kThreads), 0, stream, m.dout, shots, (uint64_t{1} << n) - 1);
        MH_HIP(hipGetLastError());
        // The uniforms are the caller's memory: the copy is complete before it returns.
        MH_HIP(hipStreamSynchronize(stream));
    }
}

ChunkedSampler::~ChunkedSampler() {
    if (impl_) (void)hipStreamSynchronize(impl_->stream);
}

uint64_t ChunkedSampler::device_bytes() const {
    return impl_->tables[0].buf.bytes() + impl_->tables[1].buf.bytes() + impl_->io.bytes();
}

void ChunkedSampler::add(const void* chunk) {
    Impl& m = *impl_;
    const uint64_t c = m.next;
    if (c >= (uint64_t{1} << (m.n - m.chunk_log))) fail(MH_ERR_INTERNAL, "chunked sampler: more chunks than the state has");
    m.next = c + 1;
    SampleArgs a = m.tables[c % 2].a;
    a.state = chunk;
    const SampleArgs& before = m.tables[(c + 1) % 2].a;
    a.carry = c == 0 ? m.zero : before.cstart + before.blocks;
    // The tables of chunk c + 2 take this slot: the stream orders them after
    // this chunk's draws and after chunk c + 1 has read the carry.
    m.tables[c % 2].a = a;
    if (m.precision == MH_C128)
        launch_tables<double2>(a, m.stream);
    else
        launch_tables<float2>(a, m.stream);
    if (m.shots == 0) return;
    if (m.precision == MH_C128)
        launch_shots<double2>(a, m.du, m.shots, m.dout, c << m.chunk_log, true, true, m.stream);
    else
        launch_shots<float2>(a, m.du, m.shots, m.dout, c << m.chunk_log, true, true, m.stream);
}

std::vector<uint64_t> ChunkedSampler::basis() {
    Impl& m = *impl_;
    if (m.next != (uint64_t{1} << (m.n - m.chunk_log))) fail(MH_ERR_INTERNAL, "chunked sampler: chunks missing");
    std::vector<uint64_t> out(m.shots);
    if (m.shots > 0) MH_HIP(hipMemcpyAsync(out.data(), m.dout, m.shots * sizeof(uint64_t), hipMemcpyDeviceToHost, m.stream));
    MH_HIP(hipStreamSynchronize(m.stream));
    return out;
}

}  // namespace mh

// A final state kept on the device with its sampler tables.
struct mh_region_sampler {
    mh::DeviceBuffer state;
    mh::SamplerTables tables;
    uint32_t n = 0;
    int32_t precision = MH_C128;
};

namespace mh {

mh_region_sampler* make_region_sampler(DeviceBuffer&& state, uint32_t n, int32_t precision) {
    amp_bytes(precision);
    if (n > 40) fail(MH_ERR_INVALID, "region sampler: num_qubits above 40");
    auto s = std::make_unique<mh_region_sampler>();
    s->state = std::move(state);
    s->n = n;
    s->precision = precision;
    if (precision == MH_C128)
        prepare_tables<double2>(s->tables, s->state.get(), n);
    else
        prepare_tables<float2>(s->tables, s->state.get(), n);
    synchronize();
    return s.release();
}

}  // namespace mh

using namespace mh;

extern "C" {

int mh_sample(const void* state, uint32_t num_qubits, int32_t precision, const double* sorted_uniforms,
              uint64_t shots, uint64_t* basis_out) {
    return guarded([&] { sample_sorted(state, num_qubits, precision, sorted_uniforms, shots, basis_out); });
}

int mh_region_sampler_draw(const mh_region_sampler* sampler, const double* uniforms, uint64_t count,
                           uint64_t* basis_out) {
    return guarded([&] {
        if (sampler == nullptr) fail(MH_ERR_INVALID, "null region sampler");
        if (count == 0) return;
        if (uniforms == nullptr || basis_out == nullptr) fail(MH_ERR_INVALID, "null uniforms or output");
        for (uint64_t i = 0; i < count; ++i)
            if (!(uniforms[i] >= 0.0 && uniforms[i] < 1.0)) fail(MH_ERR_INVALID, "region sampler: a uniform outside [0, 1)");
        if (sampler->precision == MH_C128)
            draw_basis<double2>(sampler->tables.a, uniforms, count, basis_out);
        else
            draw_basis<float2>(sampler->tables.a, uniforms, count, basis_out);
    });
}

int mh_region_sampler_info(const mh_region_sampler* sampler, uint32_t* num_qubits, uint64_t* device_bytes) {
    return guarded([&] {
        if (sampler == nullptr) fail(MH_ERR_INVALID, "null region sampler");
        if (num_qubits) *num_qubits = sampler->n;
        if (device_bytes) *device_bytes = sampler->state.bytes() + sampler->tables.buf.bytes();
    });
}

int mh_region_sampler_destroy(mh_region_sampler* sampler) {
    return guarded([&] {
        if (sampler == nullptr) return;
        synchronize();
        delete sampler;
    });
}

int mh_sample_unsorted(const void* state, uint32_t num_qubits, int32_t precision, const double* uniforms,
                       uint64_t count, uint64_t* basis_out) {
    return guarded([&] {
        std::vector<uint64_t> order(count);
        std::iota(order.begin(), order.end(), uint64_t{0});
        std::stable_sort(order.begin(), order.end(), [&](uint64_t x, uint64_t y) { return uniforms[x] < uniforms[y]; });
        std::vector<double> sorted(count);
        for (uint64_t i = 0; i < count; ++i) sorted[i] = uniforms[order[i]];
        std::vector<uint64_t> hits(count);
        sample_sorted(state, num_qubits, precision, sorted.data(), count, hits.data());
        for (uint64_t i = 0; i < count; ++i) basis_out[order[i]] = hits[i];
    });
}

}  // extern "C"

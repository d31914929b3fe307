// A resident batch replayed from a captured HIP graph (mh_batch_graph_*).
//
// The variational estimator runs the same circuits again and again with new
// parameters. The reference reruns each one from scratch (run_batch_with_options,
// src/api/batch.cpp:10-27; plan reuse by plan_job_cached /
// reparameterize_direct_plan, src/plan/plan_cache.cpp:233-276). Here the whole
// round is made resident once: fusion plans, pass programs, the state arena,
// every device table and the term-reduction descriptors; its device work is
// captured once into a graph:
//
//   matrix table <- pinned staging (copy node; it also holds each circuit's
//                   initial phase)
//   every pass of every circuit (the batch program's launches, forked over the
//   kernel streams and joined back; each circuit's first pass generates its
//   initial state, so the arena needs no clearing)
//   term reductions (kernels)
//   terms -> pinned staging (copy node)
//
// A parameter update rebuilds the block matrices and pass programs on host
// threads and writes the new matrix table into the pinned staging the graph
// copies from. How a block runs depends on its matrix (a real one leaves out its
// zero parts), so the program is built for the widest form that each block has
// had: parameters that need a narrower one (a rotation by exactly 0) run in it,
// and the first that need a wider one have the graph captured again. Only
// parameters that take a block to another class (window.h) are refused: the
// block becomes or stops being diagonal, controlled, a controlled NOT, or a
// diagonal of signs, or the first entry of a 1-qubit block real. A run is one
// graph launch. Results are the same kernels' as mh_batch_execute's, so terms
// equal it bit for bit.
#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstring>
#include <memory>
#include <string>
#include <thread>
#include <vector>

#include "batch.h"
#include "batch_program.h"
#include "engine.hpp"
#include "gate_table.h"
#include "mh_internal.h"
#include "window.h"

namespace mh {
namespace {

// Pinned host memory, freed on destruction.
class Pinned {
public:
    Pinned() = default;
    explicit Pinned(std::size_t bytes) : bytes_(bytes) {
        MH_HIP(hipHostMalloc(&ptr_, std::max<std::size_t>(bytes, 16), hipHostMallocDefault));
    }
    ~Pinned() {
        if (ptr_) (void)hipHostFree(ptr_);
    }
    Pinned(const Pinned&) = delete;
    Pinned& operator=(const Pinned&) = delete;
    Pinned(Pinned&& o) noexcept : ptr_(o.ptr_), bytes_(o.bytes_) {
        o.ptr_ = nullptr;
        o.bytes_ = 0;
    }
    Pinned& operator=(Pinned&& o) noexcept {
        if (this != &o) {
            if (ptr_) (void)hipHostFree(ptr_);
            ptr_ = o.ptr_;
            bytes_ = o.bytes_;
            o.ptr_ = nullptr;
            o.bytes_ = 0;
        }
        return *this;
    }
    void* get() const { return ptr_; }
    std::size_t bytes() const { return bytes_; }

private:
    void* ptr_ = nullptr;
    std::size_t bytes_ = 0;
};

// A circuit's structure: what its fusion plan and pass programs depend on
// besides matrix values (opcodes, qubits, parameter counts).
bool same_structure(const mh_circuit& a, const mh_circuit& b) {
    if (a.num_qubits != b.num_qubits || a.num_ops != b.num_ops) return false;
    for (uint32_t i = 0; i < a.num_ops; ++i) {
        if (a.opcodes[i] != b.opcodes[i]) return false;
        if (a.qubit_offsets[i + 1] - a.qubit_offsets[i] != b.qubit_offsets[i + 1] - b.qubit_offsets[i]) return false;
        if (a.param_offsets[i + 1] - a.param_offsets[i] != b.param_offsets[i + 1] - b.param_offsets[i]) return false;
        for (uint32_t q = a.qubit_offsets[i]; q < a.qubit_offsets[i + 1]; ++q)
            if (a.qubits[q] != b.qubits[q - a.qubit_offsets[i] + b.qubit_offsets[i]]) return false;
    }
    return true;
}

// Deep copy of a circuit's structure arrays (parameters are not kept).
struct Structure {
    std::vector<int32_t> opcodes;
    std::vector<uint32_t> qubit_offsets, qubits, param_offsets;
    mh_circuit view{};

    void copy_from(const mh_circuit& c) {
        opcodes.assign(c.opcodes, c.opcodes + c.num_ops);
        qubit_offsets.assign(c.qubit_offsets, c.qubit_offsets + c.num_ops + 1);
        qubits.assign(c.qubits, c.qubits + qubit_offsets.back());
        param_offsets.assign(c.param_offsets, c.param_offsets + c.num_ops + 1);
        view = c;
        view.opcodes = opcodes.data();
        view.qubit_offsets = qubit_offsets.data();
        view.qubits = qubits.data();
        view.param_offsets = param_offsets.data();
        view.params = nullptr;
    }
};

}  // namespace
}  // namespace mh

namespace mh {
namespace {

// A program, its tables on the device and the graph that runs it.
struct Captured {
    BatchProgram program;
    std::unique_ptr<EarlyReductions> reductions;
    DeviceBuffer bundles, ops, terms, mats, args, groups;
    Pinned pinned_mats;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    uint32_t launches = 0;

    Captured() = default;
    Captured(const Captured&) = delete;
    Captured& operator=(const Captured&) = delete;
    ~Captured() {
        if (exec) (void)hipGraphExecDestroy(exec);
        if (graph) (void)hipGraphDestroy(graph);
    }
};

}  // namespace
}  // namespace mh

struct mh_batch_graph {
    int32_t precision = MH_C128;
    int32_t fusion = MH_FUSE_CONTAINMENT;
    uint32_t fusion_width = 0;
    uint32_t max_pass_cost = 0;
    uint32_t threads = 1;
    mh::BatchSchedule schedule;
    uint32_t count = 0;
    uint32_t total_terms = 0;
    std::vector<mh::Structure> structure;
    std::vector<std::vector<mh::Block>> blocks;
    std::vector<std::vector<mh::BlockForm>> forms;  // of each block, the widest so far
    std::vector<mh::BatchItem> items;
    std::vector<uint32_t> term_offsets;
    std::vector<uint64_t> x_masks, z_masks;
    // Device residency.
    mh::DeviceBuffer arena, dterms;
    uint64_t arena_bytes = 0;
    mh::Pinned pinned_terms;
    std::unique_ptr<mh::Captured> captured;
    double plan_seconds = 0, compile_seconds = 0;
};

namespace mh {
namespace {

using clock_type = std::chrono::steady_clock;

double seconds_since(clock_type::time_point t0) {
    return std::chrono::duration<double>(clock_type::now() - t0).count();
}

// Fusion plans and block matrices of every circuit (host threads).
void plan_all(mh_batch_graph& g, const mh_circuit* circuits) {
    const auto t0 = clock_type::now();
    parallel_for(g.count, g.threads, [&](std::size_t i) {
        validate_circuit(&circuits[i]);
        const CircuitView cv{&circuits[i]};
        g.blocks[i] = build_blocks(cv, plan_fusion(cv, g.fusion, g.fusion_width));
        g.forms[i] = classify(g.blocks[i], g.precision);
    });
    g.plan_seconds = seconds_since(t0);
}

// Each item's initial phase exp(i * global_phase), from host libm.
void set_phases(std::vector<BatchItem>& items, const double* global_phases) {
    for (std::size_t i = 0; i < items.size(); ++i) {
        const std::complex<double> ph = host_phase(global_phases ? global_phases[i] : 0.0);
        items[i].initialise = true;
        items[i].phase_re = ph.real();
        items[i].phase_im = ph.imag();
    }
}

// Uploads a program's tables and captures its launches, everything on the main
// stream. A graph captured over several streams (the
// kernel streams forked off the main stream and joined back) kept the device
// memory its kernels used referenced after the graph and its executable were
// destroyed (measured on ROCm 7.2: hipFree returned success and the memory did
// not come back), so resident batches were never released; captured on one
// stream, the memory returns. One launch group at a time on one stream costs
// the default schedule nothing (it has one launch group), and the reduction
// buckets follow the launch that finishes their states.
std::unique_ptr<Captured> capture(const mh_batch_graph& g, const std::vector<BatchItem>& items, BatchProgram&& program) {
    context();
    auto c = std::make_unique<Captured>();
    c->program = std::move(program);
    auto table = [](DeviceBuffer& d, const std::vector<unsigned char>& src) {
        d = DeviceBuffer(src.size());
        upload(d.get(), src.data(), src.size());
    };
    table(c->bundles, c->program.bundles());
    table(c->ops, c->program.ops());
    table(c->terms, c->program.terms());
    table(c->args, c->program.args());
    table(c->groups, c->program.groups());
    c->mats = DeviceBuffer(c->program.mats().size());
    c->pinned_mats = Pinned(c->program.mats().size());
    std::memcpy(c->pinned_mats.get(), c->program.mats().data(), c->program.mats().size());
    if (g.total_terms > 0) {
        std::vector<ExpectationItem> terms(g.count);
        for (uint32_t i = 0; i < g.count; ++i) {
            ExpectationItem& e = terms[i];
            e.state = items[i].state;
            e.n = items[i].n;
            e.terms = g.term_offsets[i + 1] - g.term_offsets[i];
            e.x = g.x_masks.data() + g.term_offsets[i];
            e.z = g.z_masks.data() + g.term_offsets[i];
            e.out_index = g.term_offsets[i];
        }
        c->reductions = std::make_unique<EarlyReductions>(g.precision, c->program, terms, g.dterms.as<double>(), streams().main);
        c->reductions->upload(streams().copy, false);
        MH_HIP(hipStreamSynchronize(streams().copy));
    }
    synchronize();
    const hipStream_t main = streams().main;
    BatchSchedule one = g.schedule;
    one.kernel_streams = 1;
    BatchDeviceTables dev;
    dev.bundles = c->bundles.as<uint32_t>();
    dev.ops = static_cast<const WOp*>(c->ops.get());
    dev.terms = static_cast<const SignTerm*>(c->terms.get());
    dev.mats = c->mats.get();
    dev.args = static_cast<const WBatchArgs*>(c->args.get());
    dev.groups = c->groups.as<uint32_t>();
    MH_HIP(hipStreamBeginCapture(main, hipStreamCaptureModeThreadLocal));
    try {
        MH_HIP(hipMemcpyAsync(c->mats.get(), c->pinned_mats.get(), c->program.mats().size(), hipMemcpyHostToDevice, main));
        AfterLaunch after;
        if (c->reductions) after = [&](const BatchLaunch& l, hipStream_t s) { c->reductions->after(l, s); };
        c->launches = issue_batch_program(c->program, items.data(), dev, one, 0, after);
        if (c->reductions) {
            c->reductions->flush({main});
            MH_HIP(hipMemcpyAsync(g.pinned_terms.get(), g.dterms.get(), g.dterms.bytes(), hipMemcpyDeviceToHost, main));
            c->launches += c->reductions->launches();
        }
    } catch (...) {
        hipGraph_t partial = nullptr;
        (void)hipStreamEndCapture(main, &partial);
        if (partial) (void)hipGraphDestroy(partial);
        throw;
    }
    MH_HIP(hipStreamEndCapture(main, &c->graph));
    MH_HIP(hipGraphInstantiate(&c->exec, c->graph, nullptr, nullptr, 0));
    return c;
}

}  // namespace
}  // namespace mh

namespace mh {
namespace {
// New parameters (circuits of the captured structure) into the staged matrix
// table, or into a new graph where some block needs a wider form; refuses a
// change of a block's class.
void update_blocks(mh_batch_graph& g, const mh_circuit* circuits, const double* global_phases);
}  // namespace
}  // namespace mh

using namespace mh;

extern "C" {

int mh_batch_graph_create(const mh_batch_request* req, mh_batch_graph** out) {
    return guarded([&] {
        if (req == nullptr || out == nullptr) fail(MH_ERR_INVALID, "null request or output");
        *out = nullptr;
        amp_bytes(req->precision);
        if (req->num_circuits == 0 || req->circuits == nullptr || req->term_offsets == nullptr)
            fail(MH_ERR_INVALID, "a captured batch needs circuits and term offsets");
        if (req->want_statevectors) fail(MH_ERR_INVALID, "a captured batch returns terms only");
        if (req->term_offsets[0] != 0) fail(MH_ERR_INVALID, "term_offsets must start at 0");
        auto g = std::make_unique<mh_batch_graph>();
        g->precision = req->precision;
        g->fusion = req->fusion;
        g->fusion_width = req->fusion_width;
        g->max_pass_cost = req->max_pass_cost;
        g->threads = req->host_threads ? req->host_threads : std::max(1u, std::min(16u, std::thread::hardware_concurrency()));
        g->schedule.group_bytes = req->group_bytes;
        if (req->kernel_streams) g->schedule.kernel_streams = req->kernel_streams;
        g->schedule.temporal = req->cached_states != 0;
        g->count = req->num_circuits;
        g->total_terms = req->term_offsets[g->count];
        if (g->total_terms > 0 && (req->x_masks == nullptr || req->z_masks == nullptr))
            fail(MH_ERR_INVALID, "terms without masks");
        const uint32_t width = window_width(req->precision);
        g->structure.resize(g->count);
        g->blocks.resize(g->count);
        g->forms.resize(g->count);
        g->items.resize(g->count);
        g->term_offsets.assign(req->term_offsets, req->term_offsets + g->count + 1);
        uint64_t arena_bytes = 0;
        for (uint32_t i = 0; i < g->count; ++i) {
            const mh_circuit& c = req->circuits[i];
            if (c.num_qubits < width || c.num_qubits > 30)
                fail(MH_ERR_INVALID, "a batched circuit needs " + std::to_string(width) + " to 30 qubits");
            if (req->term_offsets[i + 1] < req->term_offsets[i]) fail(MH_ERR_INVALID, "term_offsets must not decrease");
            g->structure[i].copy_from(c);
            arena_bytes += round_state_bytes(c.num_qubits, req->precision);
        }
        context();
        uint64_t available = 0;
        {
            size_t free_b = 0, total_b = 0;
            MH_HIP(hipMemGetInfo(&free_b, &total_b));
            available = static_cast<uint64_t>(free_b) + pool_reusable_bytes();
        }
        if (arena_bytes > available)
            fail(MH_ERR_RESOURCE, "a captured batch keeps every state resident: " + std::to_string(arena_bytes) +
                                      " bytes, " + std::to_string(available) + " available");
        plan_all(*g, req->circuits);
        g->arena_bytes = arena_bytes;
        g->arena = DeviceBuffer(arena_bytes);
        unsigned char* base = static_cast<unsigned char*>(g->arena.get());
        if (g->total_terms > 0) {
            g->x_masks.assign(req->x_masks, req->x_masks + g->total_terms);
            g->z_masks.assign(req->z_masks, req->z_masks + g->total_terms);
            g->dterms = DeviceBuffer(uint64_t(g->total_terms) * 2 * sizeof(double));
            g->pinned_terms = Pinned(g->dterms.bytes());
        }
        uint64_t at = 0;
        for (uint32_t i = 0; i < g->count; ++i) {
            BatchItem& it = g->items[i];
            it.state = base + at;
            it.n = req->circuits[i].num_qubits;
            it.blocks = &g->blocks[i];
            it.forms = &g->forms[i];
            it.max_cost = req->max_pass_cost;
            at += round_state_bytes(it.n, req->precision);
        }
        set_phases(g->items, req->global_phases);
        const auto c0 = std::chrono::steady_clock::now();
        BatchProgram program = compile_batch_program(req->precision, g->items.data(), g->count, g->threads, g->schedule);
        g->compile_seconds = seconds_since(c0);
        if (program.has_generic() || program.needs_initialisation())
            fail(MH_ERR_INVALID, "a captured batch takes circuits with at least one gate and blocks of at most 2 "
                                 "qubits (dense) or diagonal blocks");
        g->captured = capture(*g, g->items, std::move(program));
        *out = g.release();
    });
}

int mh_batch_graph_update(mh_batch_graph* g, const mh_circuit* circuits, const double* global_phases) {
    return guarded([&] {
        if (g == nullptr || circuits == nullptr) fail(MH_ERR_INVALID, "null graph or circuits");
        for (uint32_t i = 0; i < g->count; ++i)
            if (!same_structure(circuits[i], g->structure[i].view))
                fail(MH_ERR_INVALID, "circuit " + std::to_string(i) +
                                         " differs in structure from the captured one (only parameters may change)");
        update_blocks(*g, circuits, global_phases);
    });
}

int mh_batch_graph_set_params(mh_batch_graph* g, const double* params, const double* global_phases) {
    return guarded([&] {
        if (g == nullptr) fail(MH_ERR_INVALID, "null graph");
        std::vector<mh_circuit> views(g->count);
        uint64_t at = 0;
        for (uint32_t i = 0; i < g->count; ++i) {
            views[i] = g->structure[i].view;
            const uint64_t np = views[i].param_offsets[views[i].num_ops];
            if (np > 0 && params == nullptr) fail(MH_ERR_INVALID, "null parameters");
            views[i].params = np > 0 ? params + at : nullptr;
            at += np;
        }
        update_blocks(*g, views.data(), global_phases);
    });
}

int mh_batch_graph_param_count(const mh_batch_graph* g, uint64_t* out) {
    return guarded([&] {
        if (g == nullptr || out == nullptr) fail(MH_ERR_INVALID, "null graph or output");
        uint64_t total = 0;
        for (const Structure& st : g->structure) total += st.view.param_offsets[st.view.num_ops];
        *out = total;
    });
}

}  // extern "C"

namespace mh {
namespace {

// Whether two diagonals of signs have the same ones.
bool same_signs(const Block& a, const Block& b) {
    const std::size_t dim = std::size_t{1} << a.operands.size();
    for (std::size_t e = 0; e < dim; ++e)
        if (a.matrix[e * dim + e].real() != b.matrix[e * dim + e].real()) return false;
    return true;
}

void update_blocks(mh_batch_graph& gr, const mh_circuit* circuits, const double* global_phases) {
    mh_batch_graph* g = &gr;
    std::vector<std::vector<Block>> fresh(g->count);
    std::vector<std::vector<BlockForm>> wider(g->count);  // a circuit's forms, where one got wider
    std::atomic<bool> refused{false}, again{false};
    const auto t0 = clock_type::now();
    parallel_for(g->count, g->threads, [&](std::size_t i) {
        validate_circuit(&circuits[i]);
        const CircuitView cv{&circuits[i]};
        fresh[i] = build_blocks(cv, plan_fusion(cv, g->fusion, g->fusion_width));
        const std::vector<Block>& before = g->blocks[i];
        bool ok = fresh[i].size() == before.size();
        for (std::size_t b = 0; ok && b < before.size(); ++b) ok = fresh[i][b].operands == before[b].operands;
        if (!ok) {
            refused = true;
            return;
        }
        const std::vector<BlockForm> forms = classify(fresh[i], g->precision);
        for (std::size_t b = 0; b < before.size(); ++b) {
            BlockForm f = wider[i].empty() ? g->forms[i][b] : wider[i][b];
            if (!join_form(f, forms[b], before[b].operands) ||
                (f.kind == BlockForm::kSign && !same_signs(fresh[i][b], before[b]))) {
                refused = true;
                return;
            }
            if (f == g->forms[i][b]) continue;
            if (wider[i].empty()) wider[i] = g->forms[i];
            wider[i][b] = f;
            again = true;
        }
    });
    g->plan_seconds = seconds_since(t0);
    const char* const changed =
        "the new parameters change a pass program (a matrix entry became or stopped being "
        "exactly zero or +-1); create a new captured batch for them";
    if (refused) fail(MH_ERR_INVALID, changed);
    std::vector<BatchItem> items = g->items;
    for (uint32_t i = 0; i < g->count; ++i) {
        items[i].blocks = &fresh[i];
        if (!wider[i].empty()) items[i].forms = &wider[i];
    }
    set_phases(items, global_phases);
    const auto c0 = clock_type::now();
    BatchProgram prog = compile_batch_program(g->precision, items.data(), g->count, g->threads, g->schedule);
    g->compile_seconds = seconds_since(c0);
    if (again) {
        g->captured = capture(*g, items, std::move(prog));
    } else {
        if (!prog.same_shape(g->captured->program)) fail(MH_ERR_INVALID, changed);
        std::memcpy(g->captured->pinned_mats.get(), prog.mats().data(), prog.mats().size());
        g->captured->program = std::move(prog);
    }
    g->blocks = std::move(fresh);
    for (uint32_t i = 0; i < g->count; ++i)
        if (!wider[i].empty()) g->forms[i] = std::move(wider[i]);
    g->items = std::move(items);
    for (uint32_t i = 0; i < g->count; ++i) {
        g->items[i].blocks = &g->blocks[i];
        g->items[i].forms = &g->forms[i];
    }
}

}  // namespace
}  // namespace mh

extern "C" {

int mh_batch_graph_run(mh_batch_graph* g, mh_batch_result* res) {
    return guarded([&] {
        if (g == nullptr || res == nullptr) fail(MH_ERR_INVALID, "null graph or result");
        if (g->total_terms > 0 && res->expectation_terms == nullptr) fail(MH_ERR_INVALID, "no term output");
        const auto t0 = clock_type::now();
        context();
        MH_HIP(hipGraphLaunch(g->captured->exec, streams().main));
        synchronize();
        if (g->total_terms > 0)
            std::memcpy(res->expectation_terms, g->pinned_terms.get(), uint64_t(g->total_terms) * 2 * sizeof(double));
        const double secs = seconds_since(t0);
        if (res->completion_seconds)
            for (uint32_t i = 0; i < g->count; ++i) res->completion_seconds[i] = secs;
        res->rounds = 1;
        res->launches = g->captured->launches;
        res->plan_seconds = g->plan_seconds;
        res->compile_seconds = g->compile_seconds;
        res->device_seconds = secs;
        res->total_seconds = secs;
    });
}

int mh_batch_graph_destroy(mh_batch_graph* g) {
    return guarded([&] {
        if (g == nullptr) return;
        (void)hipStreamSynchronize(streams().main);
        delete g;
    });
}

}  // extern "C"

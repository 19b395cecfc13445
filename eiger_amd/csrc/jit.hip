// jit.hip -- run-time specialisation of the row-streaming aggregation kernels.
//
// The library's hash_agg / part_agg kernels read the aggregation op list from
// their arguments (dev::RtOps), so one binary serves every request list; the
// price is per-row work on scalar loads, op-class branches and generic operand
// transforms.  For large inputs this module compiles the same kernel bodies
// (eg_agg_kernels.hpp, embedded in the library at build time) with the
// request's ops as template constants (dev::FixOps) through hipRTC, for the
// device's own architecture, and hands back the loaded function.
//
// Compilation takes about two seconds, so by default it runs on a background
// thread: calls keep using the generic kernel until the specialised one is
// ready (EG_JIT=async).  EG_JIT=sync compiles on first use; EG_JIT=off
// disables it.  Inputs below EG_JIT_MIN_ROWS rows (default 2^20) never ask for
// a specialisation.  A compile or load failure marks the entry failed and the
// generic kernel stays in use.
#include <hip/hip_runtime.h>
#include <hip/hiprtc.h>

#include <array>
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <map>
#include <memory>
#include <mutex>
#include <sstream>
#include <string>
#include <thread>
#include <unordered_map>
#include <vector>

#include "eg_internal.hpp"
#include "eg_jit.hpp"
#include "eg_lds_table.hpp"

// kJitHeaderNames / kJitHeaderTexts: the device headers, generated by the
// Makefile from the sources the library itself is built from.
#include "_build/jit_headers.inc"

namespace eg {
namespace jit {
namespace {

constexpr int kNumHeaders = (int)(sizeof(kJitHeaderNames) / sizeof(kJitHeaderNames[0]));

struct Entry {
    enum State { PENDING, READY, FAILED };
    State state = PENDING;
    std::string source;
    std::string arch;
    std::vector<char> code;
    std::string log;
    std::map<int, std::array<hipFunction_t, 2>> fn;  // per device; [1]: a hash module's storing kernel
};

struct Runtime {
    std::mutex mu;
    std::condition_variable cv;
    std::unordered_map<std::string, std::shared_ptr<Entry>> cache;
    std::deque<std::shared_ptr<Entry>> queue;
    int busy = 0;
    std::thread worker;
    bool stop = false;
    int mode = EG_JIT_ASYNC;
    int64_t min_rows = (int64_t)1 << 20;
    int64_t compiled = 0, failed = 0, launches = 0;

    Runtime()
    {
        if (const char* e = std::getenv("EG_JIT")) {
            if (!std::strcmp(e, "off") || !std::strcmp(e, "0")) mode = EG_JIT_OFF;
            else if (!std::strcmp(e, "sync")) mode = EG_JIT_SYNC;
        }
        if (const char* e = std::getenv("EG_JIT_MIN_ROWS")) min_rows = std::max<int64_t>(0, std::atoll(e));
    }
    ~Runtime()
    {
        {
            std::lock_guard<std::mutex> lk(mu);
            stop = true;
        }
        cv.notify_all();
        if (worker.joinable()) worker.join();
    }
};

Runtime& rt()
{
    static Runtime r;
    return r;
}

bool verbose()
{
    static const bool v = std::getenv("EG_JIT_VERBOSE") != nullptr;
    return v;
}

// Compiles e->source; fills code or log.  Runs without the runtime lock.
void compile(Entry* e, std::string& log, std::vector<char>& code)
{
    hiprtcProgram prog;
    if (hiprtcCreateProgram(&prog, e->source.c_str(), "eg_jit.hip", kNumHeaders, kJitHeaderTexts,
                            kJitHeaderNames) != HIPRTC_SUCCESS) {
        log = "hiprtcCreateProgram failed";
        return;
    }
    const std::string arch = "--offload-arch=" + e->arch;
    // packed fp32 forms stay off, as for the prebuilt kernels
    const char* opts[] = {arch.c_str(), "-O3", "-std=c++17", "-munsafe-fp-atomics", "-Xclang", "-target-feature",
                          "-Xclang", "-packed-fp32-ops"};
    const hiprtcResult rc = hiprtcCompileProgram(prog, (int)(sizeof(opts) / sizeof(opts[0])), opts);
    size_t ls = 0;
    if (hiprtcGetProgramLogSize(prog, &ls) == HIPRTC_SUCCESS && ls > 1) {
        log.resize(ls);
        hiprtcGetProgramLog(prog, &log[0]);
    }
    if (rc == HIPRTC_SUCCESS) {
        size_t cs = 0;
        if (hiprtcGetCodeSize(prog, &cs) == HIPRTC_SUCCESS && cs > 0) {
            code.resize(cs);
            if (hiprtcGetCode(prog, code.data()) != HIPRTC_SUCCESS) code.clear();
        }
    }
    if (code.empty() && log.empty()) log = hiprtcGetErrorString(rc);
    hiprtcDestroyProgram(&prog);
}

void finish(Runtime& r, Entry* e, std::string&& log, std::vector<char>&& code)
{
    // caller holds r.mu
    e->log = std::move(log);
    if (!code.empty()) {
        e->code = std::move(code);
        e->state = Entry::READY;
        ++r.compiled;
    } else {
        e->state = Entry::FAILED;
        ++r.failed;
        if (verbose()) std::fprintf(stderr, "eiger jit: compile failed\n%s\n", e->log.c_str());
    }
}

void join_at_exit();

// Exit handlers run in reverse order of registration, so one registered
// before a module load or a compile runs after every handler that load or
// compile registers (the runtime's and the compiler's own teardown), with the
// compile possibly still running.  The join is therefore registered again
// after each module load and before each compile: at exit it runs first, lets
// the running compile finish and joins the worker.
void arm_exit_join() { (void)std::atexit(join_at_exit); }

void worker_loop()
{
    Runtime& r = rt();
    std::unique_lock<std::mutex> lk(r.mu);
    for (;;) {
        r.cv.wait(lk, [&] { return r.stop || !r.queue.empty(); });
        if (r.stop) return;
        std::shared_ptr<Entry> e = r.queue.front();
        r.queue.pop_front();
        ++r.busy;
        lk.unlock();
        arm_exit_join();
        std::string log;
        std::vector<char> code;
        compile(e.get(), log, code);
        lk.lock();
        finish(r, e.get(), std::move(log), std::move(code));
        --r.busy;
        r.cv.notify_all();
    }
}

// Exit with the worker inside hiprtcCompileProgram crashes during static
// destruction when the compiler's own function-local statics are destroyed
// under the running compile.  A first compile in the calling thread, of a
// small kernel that still goes through the optimiser (loop, LDS, atomics),
// creates those statics before the worker exists; the exit handler (armed
// after it, and again as above) lets the in-flight compile finish, drops
// queued ones and joins the worker.  Idempotent.  One-time cost: ~0.5 s.
void join_at_exit()
{
    Runtime& r = rt();
    {
        std::lock_guard<std::mutex> lk(r.mu);
        r.stop = true;
        r.queue.clear();
    }
    r.cv.notify_all();
    if (r.worker.joinable() && r.worker.get_id() != std::this_thread::get_id()) r.worker.join();
}

void prepare_worker(const std::string& arch)
{
    static std::once_flag once;
    std::call_once(once, [&] {
        static const char* kWarmUp =
            "extern \"C\" __global__ void eg_jit_warm_up(unsigned long long* p, int n)\n"
            "{\n"
            "    __shared__ unsigned long long t[256];\n"
            "    t[threadIdx.x] = 0;\n"
            "    __syncthreads();\n"
            "    for (int i = threadIdx.x; i < n; i += blockDim.x) atomicAdd(&t[p[i] & 255], p[i] >> 8);\n"
            "    __syncthreads();\n"
            "    atomicMax(&p[threadIdx.x], t[threadIdx.x]);\n"
            "}\n";
        hiprtcProgram prog;
        if (hiprtcCreateProgram(&prog, kWarmUp, "eg_jit_warm_up.hip", 0, nullptr, nullptr) == HIPRTC_SUCCESS) {
            const std::string a = "--offload-arch=" + arch;
            const char* opts[] = {a.c_str(), "-O3"};
            (void)hiprtcCompileProgram(prog, 2, opts);
            hiprtcDestroyProgram(&prog);
        }
        arm_exit_join();
    });
}

const std::string& device_arch(int dev)
{
    static std::mutex mu;
    static std::map<int, std::string> names;
    std::lock_guard<std::mutex> lk(mu);
    auto it = names.find(dev);
    if (it == names.end()) {
        hipDeviceProp_t p{};
        EG_HIP(hipGetDeviceProperties(&p, dev));
        it = names.emplace(dev, std::string(p.gcnArchName)).first;
    }
    return it->second;
}

std::string op_list(const AggSpec& spec)
{
    std::ostringstream o;
    for (int a = 0; a < spec.nops; ++a) {
        const uint32_t w = (uint32_t)spec.ops[a].code | (uint32_t)(spec.ops[a].col + 1) << 4;
        o << (a ? ", " : "") << w << "u";
    }
    return o.str();
}

// The output columns as dev::FixOuts words (code, bytes, op, op2 + 1, is_float).
std::string out_list(const OutSpec& os)
{
    std::ostringstream o;
    for (int j = 0; j < os.nouts; ++j) {
        const OutDesc& d = os.outs[j];
        const uint32_t w = (uint32_t)d.code | (uint32_t)d.bytes << 4 | (uint32_t)d.op << 8 |
                           (uint32_t)(d.op2 + 1) << 16 | (uint32_t)(d.is_float ? 1 : 0) << 24;
        o << (j ? ", " : "") << w << "u";
    }
    return o.str();
}

bool is_hash(Kind kind) { return kind == Kind::HASH_AGG || kind == Kind::HASH_AGG_STORE; }

// The kernel's name in its module.
const char* kernel_name(Kind kind)
{
    return kind == Kind::HASH_AGG ? "eg_jit_hash_agg" : kind == Kind::HASH_AGG_STORE ? "eg_jit_hash_agg_store"
                                                                                     : "eg_jit_part_agg";
}

std::string make_source(Kind kind, int kb, const std::string& vl, const AggSpec& spec, const OutSpec* os)
{
    std::ostringstream o;
    o << "#include \"eg_agg_kernels.hpp\"\n"
      << "using JitOps = eg::dev::FixOps<" << op_list(spec) << ">;\n"
      << "using JitVL = " << vl << ";\n";
    if (!is_hash(kind))
        o << "using JitOuts = " << (os ? "eg::dev::FixOuts<" + out_list(*os) + ">" : std::string("eg::dev::RtOuts"))
          << ";\n";
    if (is_hash(kind)) {
        for (const Kind k : {Kind::HASH_AGG, Kind::HASH_AGG_STORE})
            o << "extern \"C\" __global__ __launch_bounds__(eg::agg::max_block<JitVL::NV>()) void " << kernel_name(k)
              << "(eg::KeyDesc key, int64_t n, eg::AggSpec spec, eg::GTable gt, int cr, int rep_log2, "
                 "int probe_limit, int peel_min, unsigned long long* priv)\n{\n"
              << "    eg::agg::hash_agg<" << kb << ", JitVL, JitOps, " << (k == Kind::HASH_AGG_STORE ? "true" : "false")
              << ">(key, n, spec, gt, cr, rep_log2, probe_limit, peel_min, priv);\n}\n";
    } else {
        o << "extern \"C\" __global__ __launch_bounds__(eg::agg::kPBMax, 8) void eg_jit_part_agg(eg::KeyDesc key, "
             "eg::AggSpec spec, const int64_t* perm, const eg::agg::Unit* units, eg::GTable gt, eg::OutSpec os, "
             "eg::agg::OutClaims claims, int64_t capacity, int cr, int probe, int peel_min)\n{\n"
          << "    eg::agg::part_agg<" << kb << ", JitVL, JitOps, "
          << (kind == Kind::PART_AGG_GATHER ? "true" : "false")
          << ", JitOuts>(key, spec, perm, units, gt, os, claims, capacity, cr, probe, peel_min);\n}\n";
    }
    return o.str();
}

// Queues a new cache entry on the background worker (r.mu held by lk).
void enqueue(Runtime& r, std::unique_lock<std::mutex>& lk, const std::shared_ptr<Entry>& e)
{
    r.queue.push_back(e);
    if (!r.worker.joinable()) {
        const std::string arch = e->arch;
        lk.unlock();
        prepare_worker(arch);
        lk.lock();
        if (!r.worker.joinable() && !r.stop) r.worker = std::thread(worker_loop);
    }
    r.cv.notify_all();
}

}  // namespace

hipFunction_t lookup(Kind kind, int kb, const std::string& vl, const AggSpec& spec, int64_t rows, const OutSpec* os)
{
    Runtime& r = rt();
    int dev = 0;
    EG_HIP(hipGetDevice(&dev));
    std::unique_lock<std::mutex> lk(r.mu);
    if (r.mode == EG_JIT_OFF || r.stop || rows < r.min_rows || spec.nops < 1) return nullptr;
    const std::string arch = device_arch(dev);
    std::string src = make_source(kind, kb, vl, spec, os);
    const std::string key = arch + "\n" + src;
    auto it = r.cache.find(key);
    if (it == r.cache.end()) {
        auto e = std::make_shared<Entry>();
        e->source = std::move(src);
        e->arch = arch;
        it = r.cache.emplace(key, e).first;
        if (r.mode == EG_JIT_SYNC) {
            ++r.busy;
            lk.unlock();
            std::string log;
            std::vector<char> code;
            compile(e.get(), log, code);
            lk.lock();
            finish(r, e.get(), std::move(log), std::move(code));
            --r.busy;
            r.cv.notify_all();
        } else {
            enqueue(r, lk, e);
            return nullptr;
        }
    }
    Entry* e = it->second.get();
    if (e->state != Entry::READY) return nullptr;
    const int which = kind == Kind::HASH_AGG_STORE ? 1 : 0;
    auto f = e->fn.find(dev);
    if (f != e->fn.end()) return f->second[which];
    hipModule_t mod = nullptr;
    std::array<hipFunction_t, 2> fn{};
    bool ok = hipModuleLoadData(&mod, e->code.data()) == hipSuccess;
    if (is_hash(kind))
        ok = ok && hipModuleGetFunction(&fn[0], mod, kernel_name(Kind::HASH_AGG)) == hipSuccess &&
             hipModuleGetFunction(&fn[1], mod, kernel_name(Kind::HASH_AGG_STORE)) == hipSuccess;
    else
        ok = ok && hipModuleGetFunction(&fn[0], mod, kernel_name(kind)) == hipSuccess;
    if (!ok) {
        (void)hipGetLastError();
        e->state = Entry::FAILED;
        ++r.failed;
        if (verbose()) std::fprintf(stderr, "eiger jit: module load failed on device %d\n", dev);
        return nullptr;
    }
    e->fn.emplace(dev, fn);  // modules stay loaded until the process ends
    arm_exit_join();
    return fn[which];
}

bool compile_check(Kind kind, int kb, const std::string& vl, const AggSpec& spec, const std::string& arch,
                   std::string& log, const OutSpec* os)
{
    Entry e;
    e.source = make_source(kind, kb, vl, spec, os);
    e.arch = arch;
    std::vector<char> code;
    compile(&e, log, code);
    return !code.empty();
}

bool prefetch(Kind kind, int kb, const std::string& vl, const AggSpec& spec, const std::string& arch, const OutSpec* os)
{
    Runtime& r = rt();
    std::unique_lock<std::mutex> lk(r.mu);
    if (r.mode == EG_JIT_OFF || r.stop || spec.nops < 1) return false;
    std::string src = make_source(kind, kb, vl, spec, os);
    const std::string key = arch + "\n" + src;
    if (r.cache.count(key)) return false;
    auto e = std::make_shared<Entry>();
    e->source = std::move(src);
    e->arch = arch;
    r.cache.emplace(key, e);
    enqueue(r, lk, e);
    return true;
}

bool launch(hipFunction_t f, unsigned grid, unsigned block, size_t lds, hipStream_t s, void** args)
{
    const hipError_t err = hipModuleLaunchKernel(f, grid, 1, 1, block, 1, 1, (unsigned)lds, s, args, nullptr);
    Runtime& r = rt();
    std::lock_guard<std::mutex> lk(r.mu);
    if (err != hipSuccess) {
        (void)hipGetLastError();
        // never offered again: mark every entry holding this function failed
        for (auto& kv : r.cache)
            for (auto& df : kv.second->fn)
                if (df.second[0] == f || df.second[1] == f) {
                    kv.second->state = Entry::FAILED;
                    ++r.failed;
                }
        if (verbose()) std::fprintf(stderr, "eiger jit: launch failed: %s\n", hipGetErrorString(err));
        return false;
    }
    ++r.launches;
    return true;
}

int occupancy(hipFunction_t f, int block, size_t lds)
{
    int n = 0;
    if (hipModuleOccupancyMaxActiveBlocksPerMultiprocessor(&n, f, block, lds) != hipSuccess) {
        (void)hipGetLastError();
        return 1;
    }
    return std::max(n, 1);
}

void configure(int mode, int64_t min_rows)
{
    Runtime& r = rt();
    std::lock_guard<std::mutex> lk(r.mu);
    if (mode >= EG_JIT_OFF && mode <= EG_JIT_SYNC) r.mode = mode;
    if (min_rows >= 0) r.min_rows = min_rows;
}

void wait_all()
{
    Runtime& r = rt();
    std::unique_lock<std::mutex> lk(r.mu);
    r.cv.wait(lk, [&] { return (r.queue.empty() || r.stop) && r.busy == 0; });
}

void stats(int64_t* out)
{
    Runtime& r = rt();
    std::lock_guard<std::mutex> lk(r.mu);
    out[0] = r.compiled;
    out[1] = r.failed;
    out[2] = (int64_t)r.queue.size() + r.busy;
    out[3] = r.launches;
    out[4] = r.mode;
    out[5] = r.min_rows;
}

}  // namespace jit
}  // namespace eg

// ---- C ABI -------------------------------------------------------------------------
extern "C" int eg_jit_configure(int32_t mode, int64_t min_rows)
{
    return eg::guard([&] {
        if (mode < -1 || mode > EG_JIT_SYNC) eg::raise(EG_ERR_INVALID, "eg_jit_configure: mode out of range");
        eg::jit::configure(mode, min_rows);
    });
}

extern "C" int eg_jit_wait(void)
{
    return eg::guard([&] { eg::jit::wait_all(); });
}

extern "C" int eg_jit_selftest(const char* arch, char* log, int64_t log_len)
{
    using namespace eg;
    int failures = 0;
    int st = guard([&] {
        if (!arch || !*arch) raise(EG_ERR_INVALID, "eg_jit_selftest: no architecture");
        struct Case {
            jit::Kind kind;
            int kb;
            const char* vl;
            std::vector<std::pair<int, int>> ops;  // (code, col), class-ordered
            bool outs = false;                     // compile the output list in (one column per op)
        };
        const std::vector<Case> cases = {
            {jit::Kind::HASH_AGG, 4, "eg::lds::VLayout<2, 8, 4, false, 0, 4>",
             {{OPC_COUNT, -1}, {OPC_SUM_I, 0}, {OPC_SUM_F, 1}, {OPC_MIN_I, 0}, {OPC_MAX_I, 0}}},
            {jit::Kind::PART_AGG, 4, "eg::lds::VLayout<2, 8, 4, false, 0, 4>",
             {{OPC_COUNT, -1}, {OPC_SUM_I, 0}, {OPC_SUM_F, 1}, {OPC_MIN_I, 0}, {OPC_MAX_I, 0}}},
            {jit::Kind::PART_AGG, 4, "eg::lds::VLayout<2, 8, 4, false, 0, 4>",
             {{OPC_COUNT, -1}, {OPC_SUM_I, 0}, {OPC_SUM_F, 1}, {OPC_MIN_I, 0}, {OPC_MAX_I, 0}}, true},
            {jit::Kind::HASH_AGG, 8, "eg::lds::VLayout<4, 0, 0, true, 0, 0>",
             {{OPC_SUM_U, 2}, {OPC_MAX_F, 1}, {OPC_MIN_F, 3}, {OPC_ANY, 0}}},
            {jit::Kind::PART_AGG, 8, "eg::lds::VLayout<0, 4, 4, false, 0, 0>", {{OPC_COUNT, -1}}},
            {jit::Kind::PART_AGG_GATHER, 4, "eg::lds::VLayout<1, 4, 4, false, 1, 0>", {{OPC_SUM_I, 0}, {OPC_MAX_I, 0}}},
        };
        std::string all;
        for (const Case& c : cases) {
            AggSpec spec{};
            spec.nops = (int)c.ops.size();
            for (int a = 0; a < spec.nops; ++a) {
                spec.ops[a].code = c.ops[a].first;
                spec.ops[a].col = c.ops[a].second;
            }
            OutSpec os{};
            if (c.outs) {
                static const int32_t code_of[] = {OUT_U64, OUT_U64, OUT_U64, OUT_F32, OUT_MAX_I, OUT_MIN_I};
                os.key_bytes = c.kb;
                os.nouts = spec.nops;
                for (int a = 0; a < spec.nops; ++a) {
                    const int code = c.ops[a].first;
                    os.outs[a].code = code <= OPC_MIN_I ? code_of[code] : OUT_U64;
                    os.outs[a].bytes = code == OPC_SUM_F ? 4 : 8;
                    os.outs[a].op = a;
                    os.outs[a].op2 = -1;
                    os.outs[a].is_float = code == OPC_SUM_F ? 1 : 0;
                }
            }
            std::string lg;
            if (!jit::compile_check(c.kind, c.kb, c.vl, spec, arch, lg, c.outs ? &os : nullptr)) {
                ++failures;
                all += lg + "\n";
            }
        }
        if (log && log_len > 0) {
            const size_t n = std::min<size_t>(all.size(), (size_t)log_len - 1);
            std::memcpy(log, all.data(), n);
            log[n] = 0;
        }
        if (failures) raise(EG_ERR_DEVICE, "eg_jit_selftest: " + std::to_string(failures) + " kernels failed to compile");
    });
    return st;
}

extern "C" int eg_jit_prefetch(int32_t key_type, const int32_t* val_types, int64_t num_vals,
                               const eg_agg_request* reqs, int64_t num_reqs, const char* arch, int32_t* queued)
{
    using namespace eg;
    return guard([&] {
        if (num_vals < 0 || (num_vals > 0 && !val_types)) raise(EG_ERR_INVALID, "eg_jit_prefetch: bad value types");
        // the request lowered exactly as the top-level group-by lowers it
        ViewIn key{nullptr, 0, key_type};
        std::vector<ViewIn> vals;
        for (int64_t c = 0; c < num_vals; ++c) vals.push_back(ViewIn{nullptr, 0, val_types[c]});
        const Plan plan = make_plan(&key, vals, reqs, num_reqs, false, true);
        std::string a;
        if (arch && *arch) {
            a = arch;
        } else {
            int dev = 0;
            EG_HIP(hipGetDevice(&dev));
            hipDeviceProp_t p{};
            EG_HIP(hipGetDeviceProperties(&p, dev));
            a = p.gcnArchName;
        }
        int n = 0;
        // vector-load layouts: the columns of a caller's request are 16-byte aligned
        // the output list as the partition kernel is handed it (pointers play no part)
        OutSpec os;
        void* none[kMaxOuts] = {};
        set_outspec(plan, nullptr, none, os);
        lds::with_vlayout(plan.spec, true, [&](auto vl) {
            const std::string name = jit::vlayout_name<decltype(vl)>();
            auto queue = [&](int kb) {
                n += jit::prefetch(jit::Kind::HASH_AGG, kb, name, plan.spec, a) ? 1 : 0;
                n += jit::prefetch(jit::Kind::PART_AGG, kb, name, plan.spec, a, &os) ? 1 : 0;
            };
            queue(plan.key.bytes);
            // UINT64 is what several key columns fuse into, or UINT32 where
            // their fields take at most 32 bits: ready for either
            if (key_type == EG_UINT64) queue(4);
        });
        if (queued) *queued = n;
    });
}

extern "C" int eg_jit_stats(int64_t* out6)
{
    return eg::guard([&] {
        if (!out6) eg::raise(EG_ERR_INVALID, "eg_jit_stats: null output");
        eg::jit::stats(out6);
    });
}

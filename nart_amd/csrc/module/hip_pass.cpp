// A pass over a parade as a HIP graph.  The kernels, their order and their arguments are the same at every pass, so the second
// pass is recorded while the operators run (their run functions do not know) and the later ones replay the record: one launch.
// What it gives is the host time of the launches where the host is the slower side, and the gaps between small kernels: from
// host array to host array, operator by operator -> replayed: MobileNetV2 at batch 1 161 -> 151 us, at batch 6 and 160x160 186 ->
// 179; ResNet-18 at batch 1 (129 -> 130) and ResNet-50 at batch 64 (1016 -> 1013) are level.  The second pass pays for it:
// 135 to 260 us more than the ones around it.  (A graph takes 18 - 25 us until its first kernel starts, an ordinary launch 3;
// launching the first four kernels the ordinary way in front of the graph, to hide that, gained nothing: 131.3 against 130.3 us
// for ResNet-18 at batch 1.)
//
// The first pass runs eagerly: it allocates the tensors, and a program that runs once pays nothing.  What a pass does
// beside launching - which side of a memory is current, which launches were left to a reader - is recorded as well, as the
// state it leaves behind, and restored by a replay.  A record is dropped when an operator of the workspace is prepared or
// destroyed, the workspace's stream changes, or a buffer it names has moved.
#include <algorithm>
#include <set>
#include <vector>

#include "hip_module.h"

namespace {

constexpr size_t kShortest = 8; // fewer kernels start sooner one by one (10 take 32 us as a graph, 54 one by one; 5 take 35 and 23)
constexpr long kWorth = 16;     // replays that pay for a record (155 us beside 10 a replay for MobileNetV2 at batch 1)
constexpr int kMaxWait = 256;   // eager passes before the next record, at most
constexpr int kUnread = 8;      // replays in a row that copied back an output nobody asked for

// A HIP call that may fail here without harm: its error does not stay behind for the next launch's check.
bool worked(hipError_t e)
{
    if (e != hipSuccess)
        (void)hipGetLastError();
    return e == hipSuccess;
}

// an input of the pass, as the record found it
struct PassInput {
    hip_mem_t *m;
    enum { kDevice, kMirror, kQuantized } from; // the device side; the pinned mirror (the record uploads it); quantized bytes
    const void *src, *dev;
};

// a memory that the pass writes, and the state it leaves behind
struct PassOutput {
    hip_mem_t *m;
    void *dev, *host;
    bool dev_valid, host_valid, down_issued;
    void (*pending)(void *);
    void *pending_ctx;
};

struct Pass {
    uint64_t epoch = 0;
    hipStream_t st = nullptr;
    int runs = 0;    // passes run operator by operator since the last record
    int wait = 1;    // how many of them before the next
    long served = 0; // replays of the present record
    int unread = 0;  // the last of them after which an output that the record copies back was not read
    hipGraphExec_t exec = nullptr;
    std::vector<PassInput> in;
    std::vector<PassOutput> out;
    long counted[kHipCounters] = {};

    // A program that prepares or reallocates before every few passes would record for nothing: each record that has not served
    // kWorth replays, or was refused, doubles the passes until the next attempt, one that has sets them back to one.
    void forget(bool refused = false, bool for_less = false)
    {
        if (exec) {
            HIPM_HIP(hipDeviceSynchronize()); // a replay may be under way, on a stream that may be gone
            (void)worked(hipGraphExecDestroy(exec));
        }
        if ((exec || refused) && !for_less)
            wait = served >= kWorth ? 1 : std::min(2 * wait, kMaxWait);
        exec = nullptr;
        runs = 0;
        served = unread = 0;
        in.clear();
        out.clear();
    }
};

// The null stream cannot be captured; a stream whose owner is capturing it takes the operators into that graph.
bool recordable(hipStream_t st)
{
    hipStreamCaptureStatus s = hipStreamCaptureStatusNone;
    return st != nullptr && worked(hipStreamIsCapturing(st, &s)) && s == hipStreamCaptureStatusNone;
}

// The inputs of the pass: memories that an operator reads before any has written them.  One that the host has just written and
// that a kernel uploads is uploaded by the record.  false: not a pass that can be recorded.
bool collect_inputs(Pass &p, op_t *const *ops, size_t n)
{
    std::set<const mem_t *> written, seen;
    for (size_t i = 0; i < n; ++i) {
        for (size_t k = 0; k < hip_op_activations(ops[i]); ++k) {
            mem_t *mm = ops[i]->input_tensors[k]->mem;
            if (written.count(mm))
                continue;
            if (!is_hip_mem(mm))
                return false;
            hip_mem_t *m = as_hip(mm);
            if (!seen.insert(mm).second) {
                for (const PassInput &in : p.in)
                    if (in.m == m && in.from == PassInput::kQuantized && m->q_op != ops[i])
                        return false; // read as values too: not worth a record's trouble
                continue;
            }
            hip_mem_settle(m);
            PassInput in = {m, PassInput::kDevice, nullptr, nullptr};
            if (m->q_valid && m->q_op == ops[i]) {
                in.from = PassInput::kQuantized;
                hip_mem_read_on(m, p.st);
                in.src = m->qhost, in.dev = m->qdev;
            } else if (m->host_valid && !m->dev_valid && m->host != nullptr && m->dev != nullptr && hip_mem_uploads_direct(m)) {
                in.from = PassInput::kMirror;
                hip_mem_read_on(m, p.st);
                hip_mem_use_on(m, p.st);
                in.src = m->host, in.dev = m->dev;
            } else {
                in.dev = hip_mem_dev_in(mm, p.st);
            }
            p.in.push_back(in);
        }
        for (size_t k = 0; k < ops[i]->output_size; ++k) {
            mem_t *mm = ops[i]->output_tensors[k].mem;
            if (!is_hip_mem(mm) || seen.count(mm)) // an operator writes what an earlier one reads: a view of an input
                return false;
            hip_mem_use_on(as_hip(mm), p.st); // another workspace's operators may be reading what the pass before left there
            written.insert(mm);
        }
    }
    return true;
}

void collect_outputs(Pass &p, op_t *const *ops, size_t n)
{
    std::set<hip_mem_t *> seen;
    for (size_t i = 0; i < n; ++i)
        for (size_t k = 0; k < ops[i]->output_size; ++k) {
            hip_mem_t *m = as_hip(ops[i]->output_tensors[k].mem);
            if (!seen.insert(m).second)
                continue;
            // what the host has fetched since the last record it will fetch again: the record ends with the copy
            const bool wanted = m->host_read;
            m->host_read = false;
            if (wanted && m->host != nullptr && m->host_cap >= m->size && m->dev_valid && !m->host_valid && !m->pending
                && !m->down_issued && m->size <= kHostDirect)
                hip_mem_start_download(m);
            p.out.push_back({m, m->dev, m->host, m->dev_valid, m->host_valid, m->down_issued, m->pending, m->pending_ctx});
        }
}

// Operator by operator.  What an operator may compute ahead of another's turn (conv_run_pair) it reads off the list.
void run_operators(op_t *const *ops, size_t n)
{
    hip_workspace_t *ws = reinterpret_cast<hip_workspace_t *>(ops[0]->workspace);
    ws->pass_ops = ops, ws->pass_n = n;
    for (ws->pass_at = 0; ws->pass_at < n; ++ws->pass_at)
        op_run(ops[ws->pass_at]);
    ws->pass_ops = nullptr;
}

bool record(Pass &p, op_t *const *ops, size_t n)
{
    if (!collect_inputs(p, ops, n))
        return false;
    std::vector<hip_mem_t> before_in;
    for (const PassInput &in : p.in)
        before_in.push_back(*in.m);
    long before[kHipCounters];
    for (int c = 0; c < kHipCounters; ++c)
        before[c] = *hip_counters()[c];
    if (!worked(hipStreamBeginCapture(p.st, hipStreamCaptureModeThreadLocal)))
        return false;
    run_operators(ops, n);
    collect_outputs(p, ops, n);
    hipGraph_t g = nullptr;
    size_t nodes = 0;
    bool ok = worked(hipStreamEndCapture(p.st, &g)) && g != nullptr;
    ok = ok && worked(hipGraphGetNodes(g, nullptr, &nodes)) && nodes >= kShortest;
    ok = ok && worked(hipGraphInstantiate(&p.exec, g, nullptr, nullptr, 0));
    if (g)
        (void)worked(hipGraphDestroy(g));
    for (int c = 0; c < kHipCounters; ++c) {
        p.counted[c] = *hip_counters()[c] - before[c];
        *hip_counters()[c] = before[c];
    }
    if (!ok) { // nothing of it ran: the inputs are as they were, the operators write their outputs' state again
        p.exec = nullptr;
        for (size_t i = 0; i < p.in.size(); ++i)
            *p.in[i].m = before_in[i];
    }
    return ok;
}

// everything the record names is where it was, and the inputs' contents are where it reads them
bool still_good(const Pass &p)
{
    for (const PassInput &in : p.in) {
        hip_mem_t *m = in.m;
        hip_mem_settle(m);
        if (in.from == PassInput::kQuantized) {
            if (!m->q_valid || m->qhost != in.src || m->qdev != in.dev)
                return false;
            hip_mem_read_on(m, p.st);
        } else if (in.from == PassInput::kMirror) {
            if (!m->host_valid || m->host != in.src || m->dev != in.dev)
                return false;
            hip_mem_read_on(m, p.st);
            hip_mem_use_on(m, p.st);
        } else if (hip_mem_dev_in(&m->m, p.st) != in.dev) {
            return false;
        }
    }
    for (const PassOutput &o : p.out) {
        if (o.m->dev != o.dev || (o.down_issued && o.m->host != o.host))
            return false;
        hip_mem_use_on(o.m, p.st);
    }
    return true;
}

} // namespace

bool hip_pass_run(void **state, op_t *const *ops, size_t n)
{
    static const bool off = getenv("NART_HIP_NO_GRAPH") != nullptr;
    hip_workspace_t *ws = reinterpret_cast<hip_workspace_t *>(ops[0]->workspace);
    if (off || !recordable(ws->stream))
        return false;
    ws->passes = true;
    if (*state == nullptr)
        *state = new Pass;
    Pass &p = *static_cast<Pass *>(*state);
    if (p.epoch != ws->epoch || p.st != ws->stream) {
        p.forget();
        p.epoch = ws->epoch, p.st = ws->stream;
    }
    if (p.exec != nullptr && !still_good(p))
        p.forget();
    if (p.exec != nullptr) {
        bool unread = false;
        for (const PassOutput &o : p.out)
            unread = unread || (o.down_issued && o.m->down_issued);
        p.unread = unread ? p.unread + 1 : 0;
        if (p.unread > kUnread)
            p.forget(false, true); // the next record copies back what has been read by then
    }
    if (p.exec == nullptr) {
        if (p.runs++ < p.wait) {
            run_operators(ops, n);
            return true;
        }
        if (!record(p, ops, n)) {
            p.forget(true);
            run_operators(ops, n);
            return true;
        }
    } else {
        ++p.served;
    }
    HIPM_HIP(hipGraphLaunch(p.exec, p.st));
    for (int c = 0; c < kHipCounters; ++c)
        *hip_counters()[c] += p.counted[c];
    for (const PassInput &in : p.in) {
        if (in.from == PassInput::kDevice)
            continue;
        in.m->up_pending = true, in.m->up_stream = p.st; // the pass reads pinned memory
        if (in.from == PassInput::kMirror)
            in.m->dev_valid = true, in.m->down_issued = false;
    }
    for (const PassOutput &o : p.out) {
        o.m->dev_valid = o.dev_valid, o.m->host_valid = o.host_valid, o.m->down_issued = o.down_issued, o.m->q_valid = false;
        o.m->pending = o.pending, o.m->pending_ctx = o.pending_ctx;
        ++o.m->fills;
    }
    return true;
}

void hip_pass_drop(void *state)
{
    Pass *p = static_cast<Pass *>(state);
    p->forget();
    delete p;
}

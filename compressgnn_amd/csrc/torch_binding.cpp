// `compressgnn_runtime`: the Python-visible operator module, with the operator names,
// argument order and error behaviour of the reference's extension
// (ZhengChenCS/CompressGNN src/runtime/csrc/function.cpp:9-21).  Host code only: every
// computation is a call into libcgnn_hip.so through the C ABI
// (include/compressgnn_abi.h); torch supplies tensors, the caching allocator and the
// current stream.  There is no CPU implementation behind these operators: CPU tensors
// are rejected with an error.
#include <ATen/Parallel.h>
#include <ATen/SavedTensorHooks.h>
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <hip/hip_runtime_api.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/extension.h>

#include <algorithm>
#include <array>
#include <atomic>
#include <chrono>
#include <climits>
#include <cmath>
#include <cstring>
#include <deque>
#include <functional>
#include <limits>
#include <memory>
#include <mutex>
#include <optional>
#include <sstream>
#include <map>
#include <string>
#include <thread>
#include <tuple>
#include <vector>

#include "compressgnn_abi.h"

namespace {

using torch::Tensor;

void ok(int rc, const char *what) {
    TORCH_CHECK(rc == CGNN_OK, what, ": ", cgnn_last_error());
}

cgnn_stream_t current_stream(const Tensor &t) {
    return reinterpret_cast<cgnn_stream_t>(c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream());
}

int dtype_code(const Tensor &t) {
    TORCH_CHECK(t.scalar_type() == torch::kFloat32 || t.scalar_type() == torch::kFloat64,
                "Only float32 and float64 are supported");
    return t.scalar_type() == torch::kFloat32 ? CGNN_F32 : CGNN_F64;
}

void require_gpu(const Tensor &t, const char *name) {
    TORCH_CHECK(t.is_cuda(), name, " must be a GPU tensor: this build of compressgnn_runtime has no CPU operators");
}

// Whether what is launched on this stream is recorded into a graph: contents made now exist from a replay on only.
bool capturing(const Tensor &like) {
    hipStream_t stream = reinterpret_cast<hipStream_t>(current_stream(like));
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    return stream != nullptr && hipStreamIsCapturing(stream, &status) == hipSuccess && status != hipStreamCaptureStatusNone;
}

// A lock over what the products of a block or a plan share.  The gradient of a native step runs on a thread of the
// autograd engine, without the interpreter's lock, while the program's own threads may be in another product of the
// same plan; the launches of both are ordered by their stream, the host objects behind them by this.  A thread that
// has to wait lets go of the interpreter, so that the one that holds the lock may need it (a dispatch mode's torch.empty);
// recursive for the same reason: such a mode may run a product of its own.
class Hold {
    std::unique_lock<std::recursive_mutex> lock;

public:
    explicit Hold(std::recursive_mutex &m) : lock(m, std::try_to_lock) {
        if (lock.owns_lock()) return;
        if (PyGILState_Check()) {
            pybind11::gil_scoped_release others;
            lock.lock();
        } else {
            lock.lock();
        }
    }
};

// Counters of the kernels whose last workgroup to arrive finishes a row (cgnn_csr.arrivals): every launch
// leaves them at zero, so the launches of one stream share one set, and streams, which may overlap, each have
// their own.  At most kStreams sets are held; the one used longest ago goes back to the allocator when another
// stream comes.  Under a stream capture the set belongs to the graph (its zeroing is recorded with it).
struct ArrivalPool {
    static constexpr size_t kStreams = 32;
    struct Set {
        int device;
        void *stream;
        Tensor counters;
    };
    std::deque<Set> sets;  // most recently used first
    std::mutex lock;

    Tensor get(int64_t n, const Tensor &like) {
        auto options = like.options().dtype(torch::kInt32).requires_grad(false);
        hipStream_t stream = reinterpret_cast<hipStream_t>(current_stream(like));
        if (capturing(like)) return torch::zeros({n}, options);
        std::lock_guard<std::mutex> hold(lock);
        const int device = like.device().index();
        auto it = std::find_if(sets.begin(), sets.end(), [&](const Set &s) { return s.device == device && s.stream == stream; });
        Set set{device, stream, Tensor()};
        if (it != sets.end()) {
            set = *it;
            if (it != sets.begin()) sets.erase(it);
            else if (set.counters.numel() >= n) return set.counters;
            else sets.pop_front();
        }
        if (!set.counters.defined() || set.counters.numel() < n) set.counters = torch::zeros({std::max<int64_t>(2 * n, 4096)}, options);
        sets.push_front(set);
        while (sets.size() > kStreams) sets.pop_back();
        return set.counters;
    }
};

ArrivalPool &arrival_pool() {
    static ArrivalPool *pool = new ArrivalPool();  // never destroyed: tensors must not outlive the allocator at exit
    return *pool;
}

// ----------------------------------------------------------------- CSR blocks ----

// Scratch memory of the nnz schedule (the carry rows), grown to the largest request and kept.
// A block owns one by default; the blocks of a propagation plan share one, since their
// products follow each other on one stream.  Two streams that run products over the same
// scratch at the same time would overwrite each other's carries: a caller who does that
// gives each stream a plan (or a block) of its own.
struct Scratch {
    // Held from DeviceCsr::prepare to the launch of the product: over this scratch and over the tables that the blocks
    // with this scratch make on their first product.
    std::recursive_mutex lock;
    Tensor buf;
    Tensor arrivals;  // counters that every product leaves at zero
    const Tensor &get(size_t bytes, const Tensor &like) {
        if (!buf.defined() || (size_t)buf.numel() < bytes || buf.device() != like.device())
            buf = torch::empty({(int64_t)std::max<size_t>(bytes, 1)}, like.options().dtype(torch::kUInt8));
        return buf;
    }
    Tensor captured;  // those of the product recorded last: a graph has its own and zeroes them in every replay
    int32_t *counters(int64_t n, const Tensor &like) {
        if (capturing(like)) {
            captured = torch::zeros({std::max<int64_t>(n, 1)}, like.options().dtype(torch::kInt32));
            return captured.data_ptr<int32_t>();
        }
        if (!arrivals.defined() || arrivals.numel() < n || arrivals.device() != like.device())
            arrivals = torch::zeros({std::max<int64_t>(n, 1)}, like.options().dtype(torch::kInt32));
        return arrivals.data_ptr<int32_t>();
    }
};

// A CSR block resident on the device in the layout the kernels read (int32 indices,
// row of every non-zero).  Built once per graph block.
struct DeviceCsr {
    int64_t rows = 0, cols = 0, nnz = 0;
    Tensor rowptr, colidx, rowidx, val;
    Tensor rowmap;  // optional: stored row g is output row rowmap[g]
    int64_t out_rows = 0;  // rows of the output: `rows`, or more when only the rows with entries are stored (rule levels)
    int32_t max_row_nnz = 0;
    int32_t seg_nnz = 0;
    Tensor cut_rows, empty_rows;  // the rows the runs of the nnz schedule cut / the rows without entries
    Tensor run_start;  // plain runs of the nnz schedule: where every run begins
    std::shared_ptr<Scratch> scratch = std::make_shared<Scratch>();
    // Whether AUTO may take workgroup runs, which divide long rows at other places than the nnz schedule
    // of the C ABI does (a plan's blocks do; a block on its own keeps the sums of the C ABI unless asked).
    bool workgroup_runs = false;
    // their tables made so far: one per lane layout, so a handful at most
    struct WgRuns {
        int32_t groups, len;
        Tensor table;
    };
    std::vector<WgRuns> wg_runs;
    Tensor captured_rowidx, captured_runs;  // those of the product recorded last, where they were not there before

    cgnn_csr view() const {
        cgnn_csr a{};
        a.rows = rows;
        a.cols = cols;
        a.nnz = nnz;
        a.rowptr = rowptr.data_ptr<int32_t>();
        a.colidx = nnz ? colidx.data_ptr<int32_t>() : nullptr;
        a.rowidx = (nnz && rowidx.defined()) ? rowidx.data_ptr<int32_t>() : nullptr;
        a.val = (nnz && val.defined()) ? val.data_ptr() : nullptr;
        a.max_row_nnz = max_row_nnz;
        a.seg_nnz = seg_nnz;
        a.rowmap = rowmap.defined() ? rowmap.data_ptr<int32_t>() : nullptr;
        a.run_start = run_start.defined() ? run_start.data_ptr<int32_t>() : nullptr;
        if (cut_rows.defined()) {
            a.cut_rows = cut_rows.data_ptr<int32_t>();  // a tensor without entries gives a pointer that is never read
            a.n_cut_rows = (int32_t)cut_rows.numel();
            a.empty_rows = empty_rows.data_ptr<int32_t>();
            a.n_empty_rows = (int32_t)empty_rows.numel();
        }
        return a;
    }

    // Which rows the runs cut depends on rowptr and the run length only: found once, here (two
    // small host reads at build time), so that the fix-up pass of every product goes straight to them.
    void list_rows() {
        cut_rows = Tensor();
        empty_rows = Tensor();
        if (rows == 0 || nnz == 0) return;
        cgnn_csr a = view();
        const int64_t K = cgnn_spmm_run_length(&a);
        Tensor start = rowptr.slice(0, 0, rows).to(torch::kInt64), end = rowptr.slice(0, 1, rows + 1).to(torch::kInt64);
        // a row of at most K entries is never cut; a longer one is cut at the multiples of K inside it
        Tensor cut = ((end - start) > K).logical_and((torch::floor_divide(start, K) + 1) * K < end);
        Tensor found = torch::nonzero(cut).flatten().to(torch::kInt32);
        Tensor none = torch::nonzero(start == end).flatten().to(torch::kInt32);
        // a pointer is needed even for an empty list (NULL means "no lists"): keep one entry of storage
        auto pad = [](const Tensor &t) { return t.numel() ? t : torch::zeros({1}, t.options()).narrow(0, 0, 0); };
        cut_rows = pad(found.contiguous());
        empty_rows = pad(none.contiguous());
    }

    // The block as a product of width F reads it, and the scratch for that product; the caller holds scratch->lock until
    // the product is launched.
    // What the nnz schedule reads beside the block is made when a product first resolves to it, on the product's
    // stream: rowidx (the row of every non-zero, as large as colidx), and the run starts of the plain runs or the table of
    // the workgroup runs for a lane layout.  Recorded into a graph they are the graph's, which fills them with every replay:
    // there is nothing in them before, so no eager product may find them.
    cgnn_csr prepare(int64_t F, int dtype, int kernel, void **ws, size_t *bytes) {
        cgnn_csr a = view();
        if (nnz > 0 && cgnn_spmm_schedule(rows, nnz, max_row_nnz, kernel) == CGNN_SPMM_NNZ) {
            const auto stream = current_stream(rowptr);
            const bool recorded = capturing(rowptr);
            if (!rowidx.defined()) {
                Tensor made = torch::empty({nnz}, rowptr.options());
                ok(cgnn_csr_expand_rows(rows, nnz, rowptr.data_ptr<int32_t>(), made.data_ptr<int32_t>(), stream), "csr_expand_rows");
                a.rowidx = made.data_ptr<int32_t>();
                (recorded ? captured_rowidx : rowidx) = made;
            }
            if (workgroup_runs && kernel == CGNN_SPMM_AUTO && empty_rows.defined()) {
                int64_t arrivals = 0;
                ok(cgnn_spmm_wg_shape(&a, F, dtype, &a.wg_groups, &a.wg_len, &arrivals), "spmm_wg_shape");
                auto found = std::find_if(wg_runs.begin(), wg_runs.end(), [&](const WgRuns &r) {
                    return r.groups == a.wg_groups && r.len == a.wg_len;
                });
                if (found == wg_runs.end()) {
                    Tensor table = torch::empty({(nnz + a.wg_len - 1) / a.wg_len * a.wg_groups + 1}, rowptr.options());
                    ok(cgnn_spmm_wg_runs(&a, a.wg_groups, a.wg_len, table.data_ptr<int32_t>(), stream), "spmm_wg_runs");
                    if (recorded) captured_runs = table;
                    else found = wg_runs.insert(wg_runs.end(), WgRuns{a.wg_groups, a.wg_len, table});
                }
                a.wg_runs = (found != wg_runs.end() ? found->table : captured_runs).data_ptr<int32_t>();
                a.arrivals = scratch->counters(arrivals, rowptr);
            } else if (!run_start.defined()) {
                const int64_t K = cgnn_spmm_run_length(&a);
                Tensor starts = torch::empty({(nnz + K - 1) / K + 1}, rowptr.options());
                ok(cgnn_spmm_run_starts(&a, starts.data_ptr<int32_t>(), stream), "spmm_run_starts");
                a.run_start = starts.data_ptr<int32_t>();
                (recorded ? captured_runs : run_start) = starts;
            }
        }
        *bytes = cgnn_spmm_workspace_bytes(&a, F, dtype, kernel);
        *ws = *bytes ? scratch->get(*bytes, rowptr).data_ptr() : nullptr;
        return a;
    }
};

// A tensor of the block that a product on another thread may be making.
Tensor locked(DeviceCsr &A, Tensor DeviceCsr::*made) {
    const std::shared_ptr<Scratch> scratch = A.scratch;
    Hold hold(scratch->lock);
    return A.*made;
}

// rowptr/col: int64 or int32 tensors on any device; value: float tensor or undefined.
std::shared_ptr<DeviceCsr> make_csr(Tensor rowptr, Tensor col, c10::optional<Tensor> value, int64_t rows,
                                    int64_t cols, torch::Device device, int64_t seg_nnz,
                                    c10::optional<Tensor> rowmap = c10::nullopt, bool with_row_lists = true,
                                    int64_t out_rows = -1) {
    TORCH_CHECK(device.is_cuda(), "DeviceCsr lives on a GPU");
    TORCH_CHECK(rowptr.dim() == 1 && col.dim() == 1 && rowptr.numel() == rows + 1, "rowptr must have rows+1 entries");
    auto blk = std::make_shared<DeviceCsr>();
    blk->rows = rows;
    blk->out_rows = out_rows < 0 ? rows : out_rows;
    TORCH_CHECK(blk->out_rows >= rows && (blk->out_rows == rows || (rowmap.has_value() && rowmap->defined())),
                "a block that stores fewer rows than its output has needs a rowmap");
    blk->cols = cols;
    blk->nnz = col.numel();
    blk->seg_nnz = (int32_t)seg_nnz;
    const int64_t lim = (int64_t)INT32_MAX - 65536;
    TORCH_CHECK(rows < lim && cols < lim && blk->nnz < lim, "block exceeds the int32 index range of the kernels");
    c10::hip::HIPGuardMasqueradingAsCUDA guard(device);
    Tensor rp = rowptr.to(device).contiguous();
    Tensor ci = col.to(device).contiguous();
    auto i32 = torch::TensorOptions().device(device).dtype(torch::kInt32);
    if (rp.scalar_type() == torch::kInt64) {
        blk->rowptr = torch::empty({rows + 1}, i32);
        blk->colidx = torch::empty({blk->nnz}, i32);
        TORCH_CHECK(ci.scalar_type() == torch::kInt64, "rowptr and col must have the same integer type");
        ok(cgnn_csr_prepare_i64(rows, blk->nnz, rp.data_ptr<int64_t>(), blk->nnz ? ci.data_ptr<int64_t>() : nullptr,
                                blk->rowptr.data_ptr<int32_t>(), blk->nnz ? blk->colidx.data_ptr<int32_t>() : nullptr,
                                nullptr, current_stream(rp)),
           "csr_prepare");
    } else {
        TORCH_CHECK(rp.scalar_type() == torch::kInt32 && ci.scalar_type() == torch::kInt32,
                    "rowptr/col must be int64 or int32");
        blk->rowptr = rp;
        blk->colidx = ci;
    }
    if (value.has_value() && value->defined()) {
        TORCH_CHECK(value->numel() == blk->nnz, "value must have one entry per non-zero");
        blk->val = value->to(device).contiguous();
    }
    if (rowmap.has_value() && rowmap->defined()) {
        TORCH_CHECK(rowmap->dim() == 1 && rowmap->numel() == rows, "rowmap must have one entry per row");
        blk->rowmap = rowmap->to(device).to(torch::kInt32).contiguous();
    }
    if (rows > 0) {
        // one host read per block, at build time: the longest row, and which entries of the arrays the rows hold
        Tensor lens = blk->rowptr.slice(0, 1, rows + 1) - blk->rowptr.slice(0, 0, rows);
        Tensor found = torch::stack({lens.max(), blk->rowptr[0], blk->rowptr[rows]}).cpu();
        blk->max_row_nnz = found.data_ptr<int32_t>()[0];
        const int64_t first = found.data_ptr<int32_t>()[1], held = found.data_ptr<int32_t>()[2] - first;
        if (first != 0 || held != blk->nnz) {
            // a slice of a larger block's row pointers, or a list that is padded behind its last row: the schedules
            // deal the entries 0 ... nnz, so the block keeps the ones in use and counts from the first of them
            TORCH_CHECK(held == 0 || (first >= 0 && held > 0 && first + held <= blk->nnz),
                        "rowptr names entries that col does not have");
            blk->rowptr = blk->rowptr - first;
            blk->colidx = blk->colidx.narrow(0, held == 0 ? 0 : first, held).clone();
            if (blk->val.defined()) blk->val = blk->val.narrow(0, held == 0 ? 0 : first, held).clone();
            blk->nnz = held;
        }
    }
    if (with_row_lists) blk->list_rows();
    return blk;
}

int kernel_of_method(const std::string &method) {
    // The reference's GPU method strings (src/runtime/csrc/sparse/cuda/spmm_gpu.cu:27-31) and
    // its two CPU ones are accepted.  Its layers pick among them from (nnz, width) alone
    // (layer/CompressgnnSPMM.py:14-19) and, for instance, ask for "rowbalance_rowcache" on every
    // large block, power-law in-lists included, where a lane group per row is many times slower
    // here.  They are therefore hints: the schedule is chosen from the block's row lengths, as
    // for "auto".  "row_schedule" and "nnz_schedule" are this build's names for a forced
    // schedule (bit-exact comparisons with a sequential sum, measurements).
    static const char *const hints[] = {"auto", "rowbalance", "rowbalance_parreduce", "rowbalance_seqreduce",
                                        "rowbalance_rowcache", "nnzbalance", "nnzbalance_parreduce",
                                        "nnzbalance_seqreduce", "nnzbalance_rowcache"};
    for (const char *h : hints)
        if (method == h) return CGNN_SPMM_AUTO;
    if (method == "row_schedule") return CGNN_SPMM_ROW;
    if (method == "nnz_schedule") return CGNN_SPMM_NNZ;
    TORCH_CHECK(false, "Invalid SpMM method: ", method);
}

// out (+)= A * mat.  `out` undefined: a fresh [rows, F] tensor is returned.
Tensor block_spmm(DeviceCsr &A, const Tensor &mat, c10::optional<Tensor> optional_out, int kernel) {
    require_gpu(mat, "mat");
    TORCH_CHECK(mat.is_contiguous(), "mat must be contiguous");
    TORCH_CHECK(mat.dim() == 2, "mat must be a matrix");
    TORCH_CHECK(mat.size(0) == A.cols, "mat has ", mat.size(0), " rows, the block has ", A.cols, " columns");
    TORCH_CHECK(!A.val.defined() || A.val.scalar_type() == mat.scalar_type(), "value and mat must have the same dtype");
    c10::hip::HIPGuardMasqueradingAsCUDA guard(mat.device());
    const int64_t F = mat.size(1);
    const int dtype = dtype_code(mat);
    Tensor out;
    int accumulate = 0;
    if (optional_out.has_value() && optional_out->defined()) {
        // like the reference (spmm_gpu.cu:20-22) a non-contiguous out is copied, so the
        // caller must use the returned tensor
        out = optional_out->contiguous();
        require_gpu(out, "out");
        TORCH_CHECK(out.dim() == 2 && out.size(0) == A.out_rows && out.size(1) == F && out.scalar_type() == mat.scalar_type(),
                    "out must be [rows, F] of mat's dtype");
        accumulate = 1;
    } else if (A.out_rows != A.rows) {
        out = torch::zeros({A.out_rows, F}, mat.options());  // the rows that are not stored have no entries
    } else {
        out = torch::empty({A.rows, F}, mat.options());
    }
    if (A.rows == 0 || F == 0) return out;
    size_t bytes = 0;
    void *ws = nullptr;
    const std::shared_ptr<Scratch> scratch = A.scratch;
    Hold hold(scratch->lock);
    cgnn_csr a = A.prepare(F, dtype, kernel, &ws, &bytes);
    ok(cgnn_spmm(&a, dtype, mat.data_ptr(), out.data_ptr(), F, accumulate, kernel, ws, bytes,
                 current_stream(mat)),
       "spmm");
    return out;
}

// spmm_func of the reference (src/runtime/csrc/sparse/spmm.cpp:11-22): CSR given as
// int64 tensors, whose rows are looked for on every call.  Graph blocks that are used repeatedly should
// be wrapped in a DeviceCsr once instead.
Tensor spmm_func(Tensor vlist, Tensor elist, Tensor value, Tensor mat, std::string method,
                 c10::optional<Tensor> optional_out) {
    require_gpu(mat, "mat");
    require_gpu(vlist, "vlist");
    require_gpu(elist, "elist");
    require_gpu(value, "value");
    const int kernel = kernel_of_method(method);
    TORCH_CHECK(vlist.scalar_type() == torch::kInt64 && elist.scalar_type() == torch::kInt64,
                "vlist and elist must be int64");
    const int64_t rows = vlist.size(-1) - 1, nnz = elist.numel();
    const bool plain = mat.dim() == 2 && mat.is_contiguous() && vlist.dim() == 1 && elist.dim() == 1 && rows > 0 && nnz > 0 &&
                       mat.size(1) > 0 && vlist.device() == mat.device() && elist.device() == mat.device() &&
                       value.device() == mat.device();
    if (kernel != CGNN_SPMM_AUTO || !plain) {
        auto blk = make_csr(vlist, elist, value, rows, mat.size(0), mat.device(), 0, c10::nullopt, false);
        return block_spmm(*blk, mat, optional_out, kernel);
    }
    const int64_t F = mat.size(1), lim = (int64_t)INT32_MAX - 65536;
    TORCH_CHECK(rows < lim && mat.size(0) < lim && nnz < lim, "block exceeds the int32 index range of the kernels");
    TORCH_CHECK(value.numel() == nnz, "value must have one entry per non-zero");
    TORCH_CHECK(value.scalar_type() == mat.scalar_type(), "value and mat must have the same dtype");
    c10::hip::HIPGuardMasqueradingAsCUDA guard(mat.device());
    const int dtype = dtype_code(mat);
    const Tensor rowptr = vlist.contiguous(), col = elist.contiguous(), val = value.contiguous();
    Tensor out;
    const bool accumulate = optional_out.has_value() && optional_out->defined();
    if (accumulate) {
        out = optional_out->contiguous();  // as in block_spmm
        require_gpu(out, "out");
        TORCH_CHECK(out.dim() == 2 && out.size(0) == rows && out.size(1) == F && out.scalar_type() == mat.scalar_type(),
                    "out must be [rows, F] of mat's dtype");
    } else {
        out = torch::empty({rows, F}, mat.options());
    }
    int64_t arrivals = 0;
    const size_t bytes = cgnn_spmm_once_workspace_bytes(rows, nnz, F, dtype, &arrivals);
    Tensor ws = torch::empty({(int64_t)bytes}, mat.options().dtype(torch::kUInt8));
    Tensor counters = arrival_pool().get(arrivals, mat);
    ok(cgnn_spmm_once(rows, nnz, rowptr.data_ptr<int64_t>(), col.data_ptr<int64_t>(), val.data_ptr(), dtype, mat.data_ptr(),
                      out.data_ptr(), F, accumulate, ws.data_ptr(), bytes, counters.data_ptr<int32_t>(), current_stream(mat)),
       "spmm");
    return out;
}

// ------------------------------------------------------- compressed propagation ----

// Optional per-stage timing with HIP events on the stream the kernels run on.  Events
// are recorded only around the stages named in `timed` ("*" = all), so a timed region
// can carry one pair of events per step without disturbing the rest.
struct StageTimer {
    struct Rec {
        std::string name;
        hipEvent_t begin, end;
    };
    std::vector<std::string> timed;
    std::vector<Rec> recs;
    // An event pair costs the stream a few microseconds of idle time on either side of the stage, so
    // a caller that times a loop may ask for every n-th pass of a stage only.
    int64_t every = 1;
    std::map<std::string, int64_t> passes;

    bool wants(const std::string &name) const {
        for (auto &t : timed)
            if (t == "*" || t == name) return true;
        return false;
    }
    int open(const std::string &name, hipStream_t stream) {
        if (!wants(name)) return -1;
        if (passes[name]++ % std::max<int64_t>(every, 1) != 0) return -1;
        Rec r{name, nullptr, nullptr};
        TORCH_CHECK(hipEventCreate(&r.begin) == hipSuccess && hipEventCreate(&r.end) == hipSuccess, "hipEventCreate failed");
        TORCH_CHECK(hipEventRecord(r.begin, stream) == hipSuccess, "hipEventRecord failed");
        recs.push_back(r);
        return (int)recs.size() - 1;
    }
    void close(int id, hipStream_t stream) {
        if (id >= 0) TORCH_CHECK(hipEventRecord(recs[id].end, stream) == hipSuccess, "hipEventRecord failed");
    }
    // (stage, milliseconds) of every recorded interval; call after the stream is idle.
    std::vector<std::pair<std::string, double>> take() {
        std::vector<std::pair<std::string, double>> out;
        for (auto &r : recs) {
            float ms = 0;
            TORCH_CHECK(hipEventSynchronize(r.end) == hipSuccess, "hipEventSynchronize failed");
            TORCH_CHECK(hipEventElapsedTime(&ms, r.begin, r.end) == hipSuccess, "hipEventElapsedTime failed");
            out.emplace_back(r.name, (double)ms);
            hipEventDestroy(r.begin);
            hipEventDestroy(r.end);
        }
        recs.clear();
        return out;
    }
    ~StageTimer() {
        for (auto &r : recs) {
            hipEventDestroy(r.begin);
            hipEventDestroy(r.end);
        }
    }
};

// What a multiplied-out block is made of, by version counter: the columns and values of a vertex stage and its rules.
// They may be tensors of the caller's (DeviceCsr takes int32 and float arrays as they are), and the stages read them
// with every product.  Writes to inference tensors are not counted; those are taken as they were.
std::array<uint32_t, 4> written(const DeviceCsr &stage, const DeviceCsr &rules) {
    auto version = [](const Tensor &t) { return t.defined() && !t.is_inference() ? (uint32_t)t._version() : 0u; };
    return {version(stage.colidx), version(stage.val), version(rules.colidx), version(rules.val)};
}

// A vertex stage with its rules multiplied out ([vertex_cnt, vertex_cnt], the same stored rows): a propagation in one
// launch where the compressed form does not save what its second launch costs (takes_whole).
struct MultipliedOut {
    int64_t entries = 0;  // 0: never
    int32_t longest = 0;  // its longest row
    Tensor starts;        // its row pointers
    std::array<uint32_t, 4> made_of{};
    std::shared_ptr<DeviceCsr> block;  // made for the first product that takes it
};

// The device form of a CompressGraph (loader/compress_graph.py:6-43 of the reference):
// the three vertex/rule blocks, the rule levels and their transposes.
struct PropagationPlan {
    // rule stage and rule levels, forward and backward
    std::shared_ptr<DeviceCsr> r2v, v2r_t;
    std::vector<std::shared_ptr<DeviceCsr>> r2r, r2r_t;
    // [v2v | v2r] and [v2v^T | r2v^T]: the vertex stage of forward / backward in one pass
    std::shared_ptr<DeviceCsr> vertex_stage, vertex_stage_t;
    MultipliedOut whole, whole_t;
    // the four blocks of the vertex stages on their own: only for the two-launch form
    // (fuse_final = false); a plan without them holds its stages once
    std::shared_ptr<DeviceCsr> v2v, v2r, v2v_t, r2v_t;
    int64_t V = 0, R = 0;
    bool fuse_final = true;  // last two stages in one pass (cgnn_spmm_dual)
    int kernel = CGNN_SPMM_AUTO;
    std::shared_ptr<Scratch> scratch = std::make_shared<Scratch>();
    std::recursive_mutex lock;  // held for a chain of products: over the timer and the composed blocks
    StageTimer timer;
    // The forward blocks with their vertex columns sent through a cluster assignment
    // (propagate_forward_gathered), kept for the index tensors they were made for: an
    // assignment lasts until the next refresh, and a model may hold one per layer.  Either form, or both, as products ask.
    struct Composed {
        c10::weak_intrusive_ptr<c10::TensorImpl> index;
        uint32_t version;
        int64_t groups;
        std::shared_ptr<DeviceCsr> rules, stage, whole;
    };
    std::deque<std::shared_ptr<Composed>> composed;

    void adopt(const std::shared_ptr<DeviceCsr> &block) {
        if (!block) return;
        block->scratch = scratch;
        block->workgroup_runs = true;
    }
    bool fused() const { return fuse_final && vertex_stage && vertex_stage_t; }
    void require_split_blocks() const {
        TORCH_CHECK(v2v && v2r && v2v_t && r2v_t,
                    "this plan holds the fused vertex stages only; the two-launch form needs the v2v, v2r, v2v_t and "
                    "r2v_t blocks (graph.keep_split_blocks = True before graph.plan())");
    }
};

// A propagation with the rules multiplied out.  The rule stage is a launch that the vertex stage waits for: 3 to 12 us
// however few entries it holds, 20 where the few rules of a small graph have long rows.  Multiplied out, the vertex stage
// is a launch alone and gathers what the rules had saved it; on web graphs of 20,000 to 325,557 vertices both
// forms take the same time where that is 45 to 60 MB more than the two stages move, and 75 to 90 MB in the row schedule,
// whose stored neighbours share most of what they gather (forward + gradient, us, two stages against one: 64 features over
// 2,708 vertices 25 / 16, 10,000 41 / 14, 50,001 49 / 37, 100,003 81 / 69, 200,000 of degree 5 100 / 89; beyond the line
// 128 features over 325,557 vertices 365 / 388).
constexpr int64_t kRuleStageBytes = int64_t(48) << 20, kRuleStageBytesRowSchedule = int64_t(72) << 20;

// No more entries than this are kept beside the stages: beyond, a propagation takes so long that a launch is nothing to
// it, and the device would hold a large graph twice.
constexpr int64_t kMaxWholeEntries = int64_t(1) << 22;

// Whether a product whose rows take row_bytes is as fast with the `entries` of the multiplied-out stage.
bool takes_whole(int64_t entries, const DeviceCsr &stage, const DeviceCsr &rules, int64_t row_bytes) {
    const int64_t index_bytes = 12;  // column, value, row
    const int64_t more = (entries - stage.nnz - rules.nnz) * (row_bytes + index_bytes) - 2 * rules.rows * row_bytes;
    const bool row_schedule = cgnn_spmm_schedule(stage.rows, stage.nnz, stage.max_row_nnz, CGNN_SPMM_AUTO) == CGNN_SPMM_ROW;
    return more <= (row_schedule ? kRuleStageBytesRowSchedule : kRuleStageBytes);
}

// Whether every product of a value that stands for a rule and a value of the rules has a place in the type T, by the
// extremes of both (cgnn_csr_expand_summary).  A multiplied-out block stores these products; the stages multiply through
// the sums of the rules, and factors like 1e-25 and 1e-25, or 1e25 and 1e25, are theirs.
template <typename T>
bool products_in_range(const uint64_t *magnitudes) {
    long double of[4];
    for (int k = 0; k < 4; ++k) {
        if (magnitudes[k] == UINT64_MAX) return true;  // all zero, or none
        T v;
        std::memcpy(&v, &magnitudes[k], sizeof(T));  // the low half comes first
        of[k] = v;
    }
    return std::isfinite(of[0]) && std::isfinite(of[2]) && of[0] * of[2] <= std::numeric_limits<T>::max() &&
           of[1] * of[3] >= std::numeric_limits<T>::min();
}

// The block as a kernel reads it, beside a product on another thread that makes tables of it.
cgnn_csr viewed(const DeviceCsr &A) {
    const std::shared_ptr<Scratch> scratch = A.scratch;
    Hold hold(scratch->lock);
    return A.view();
}

// What the vertex stages [vertices | rules] of both directions come to with their rules multiplied out; no entries where no
// product would take that, or a value has no place in it.  One host read.
std::array<MultipliedOut, 2> surveyed(const std::array<std::pair<DeviceCsr *, DeviceCsr *>, 2> &stages, int64_t V) {
    std::array<MultipliedOut, 2> found;
    const Tensor like = stages[0].first->rowptr;
    if (capturing(like)) return found;
    c10::hip::HIPGuardMasqueradingAsCUDA guard(like.device());
    const auto stream = current_stream(like);
    Tensor summaries, starts[2];
    bool wanted[2];
    uint64_t empty[2] = {0, 0};
    for (int k = 0; k < 2; ++k) {
        const DeviceCsr &stage = *stages[k].first, &rules = *stages[k].second;
        const Tensor empty_rows = locked(*stages[k].first, &DeviceCsr::empty_rows);
        wanted[k] = empty_rows.defined() && rules.nnz > 0 && stage.val.defined() && stage.nnz <= kMaxWholeEntries &&
                    (stage.val.scalar_type() == torch::kFloat32 || stage.val.scalar_type() == torch::kFloat64) &&
                    (!rules.val.defined() || rules.val.scalar_type() == stage.val.scalar_type()) &&
                    stage.rowptr.device() == like.device() && rules.rowptr.device() == like.device();
        if (!wanted[k]) continue;
        empty[k] = (uint64_t)empty_rows.numel();
        found[k].made_of = written(stage, rules);
        if (!summaries.defined()) summaries = torch::empty({2, CGNN_EXPAND_SUMMARY}, like.options().dtype(torch::kInt64));
        const cgnn_csr a = viewed(stage), r = viewed(rules);
        Tensor counts = torch::empty({stage.rows}, like.options());
        ok(cgnn_csr_expand_count(&a, V, &r, counts.data_ptr<int32_t>(), stream), "csr_expand_count");
        ok(cgnn_csr_expand_summary(&a, V, &r, dtype_code(stage.val), counts.data_ptr<int32_t>(),
                                   reinterpret_cast<uint64_t *>(summaries[k].data_ptr<int64_t>()), stream),
           "csr_expand_summary");
        starts[k] = torch::empty({stage.rows + 1}, like.options());
        const size_t bytes = cgnn_exclusive_sum_workspace_bytes(stage.rows);
        Tensor ws = torch::empty({(int64_t)bytes}, like.options().dtype(torch::kUInt8));
        ok(cgnn_exclusive_sum_i32(stage.rows, counts.data_ptr<int32_t>(), starts[k].data_ptr<int32_t>(), nullptr, ws.data_ptr(), bytes, stream),
           "exclusive_sum");
    }
    if (!summaries.defined()) return found;
    summaries = summaries.cpu();
    for (int k = 0; k < 2; ++k) {
        if (!wanted[k]) continue;
        const uint64_t *s = reinterpret_cast<const uint64_t *>(summaries.data_ptr<int64_t>()) + k * CGNN_EXPAND_SUMMARY;
        const DeviceCsr &stage = *stages[k].first;
        const bool in_range = stage.val.scalar_type() == torch::kFloat32 ? products_in_range<float>(s + 3) : products_in_range<double>(s + 3);
        // (a row that only rules without entries stand in would be one that the stage's list of empty rows does not have)
        if (s[0] > (uint64_t)kMaxWholeEntries || s[2] != empty[k] || !in_range) continue;
        found[k].entries = (int64_t)s[0];
        found[k].longest = (int32_t)s[1];
        found[k].starts = starts[k];
    }
    return found;
}

// Waits for the stream; the interpreter's other threads run meanwhile.
bool synchronized(cgnn_stream_t stream) {
    auto wait = [&] { return hipStreamSynchronize(reinterpret_cast<hipStream_t>(stream)) == hipSuccess; };
    if (!PyGILState_Check()) return wait();
    pybind11::gil_scoped_release others;
    return wait();
}

// The multiplied-out stage where a product with x takes it, else NULL.  A forced schedule and the two-launch form run the
// stages, and so does every product once one of their arrays was written to.  (A graph replays what it recorded: after such a
// write it has to be captured again.)  Made for the first product that takes it, so that a plan whose products are all wide
// holds the graph once, and finished when that product is launched, whatever stream the next one runs on; no array
// needs a host read to be made, so under a capture it is the graph's, which makes it with every replay (a program that runs a
// product first captures the finished one).  The caller holds the plan's lock.
std::shared_ptr<DeviceCsr> multiplied_out(PropagationPlan &p, MultipliedOut &whole, const std::shared_ptr<DeviceCsr> &stage,
                                          const std::shared_ptr<DeviceCsr> &rules, const Tensor &x) {
    if (whole.entries == 0 || !p.fuse_final || p.kernel != CGNN_SPMM_AUTO || x.scalar_type() != stage->val.scalar_type() ||
        x.size(1) == 0 || x.device() != stage->rowptr.device() ||
        !takes_whole(whole.entries, *stage, *rules, x.size(1) * x.element_size()))
        return nullptr;
    if (whole.made_of != written(*stage, *rules)) {
        whole.entries = 0;  // the block stays until the plan goes: a product on another stream may still read it
        return nullptr;
    }
    if (whole.block) return whole.block;
    const auto stream = current_stream(x);
    const auto ints = stage->rowptr.options();
    auto blk = std::make_shared<DeviceCsr>();
    blk->rows = blk->out_rows = stage->rows;
    blk->cols = p.V;
    blk->nnz = whole.entries;
    blk->max_row_nnz = whole.longest;
    blk->seg_nnz = stage->seg_nnz;
    blk->rowmap = stage->rowmap;
    blk->rowptr = whole.starts;
    // A graph that recorded the making may be replayed after the columns were written to, and rows then come to more or fewer
    // entries than they have room for: they are cut off, or keep entries (0, 0), so that the arrays are the block that the
    // starts say whatever the columns are, and no product reads or writes outside them.
    blk->colidx = torch::zeros({whole.entries}, ints);
    blk->val = torch::zeros({whole.entries}, stage->val.options());
    // The plan's AUTO products run the row schedule or workgroup runs: neither asks which rows plain runs would cut.
    blk->cut_rows = torch::empty({1}, ints).narrow(0, 0, 0);
    blk->empty_rows = locked(*stage, &DeviceCsr::empty_rows);
    p.adopt(blk);
    const cgnn_csr a = viewed(*stage), r = viewed(*rules);
    ok(cgnn_csr_expand_columns(&a, p.V, &r, dtype_code(x), blk->rowptr.data_ptr<int32_t>(), blk->colidx.data_ptr<int32_t>(),
                               blk->val.data_ptr(), stream),
       "csr_expand_columns");
    if (capturing(x)) return blk;
    TORCH_CHECK(synchronized(stream), "propagate: the stream reported an error");
    whole.block = blk;
    return blk;
}

Tensor timed_spmm(PropagationPlan &p, const std::string &stage, DeviceCsr &A, const Tensor &mat,
                  c10::optional<Tensor> out) {
    hipStream_t stream = reinterpret_cast<hipStream_t>(current_stream(mat));
    const int id = p.timer.open(stage, stream);
    Tensor r = block_spmm(A, mat, out, p.kernel);
    p.timer.close(id, stream);
    return r;
}

Tensor final_stage(PropagationPlan &p, const std::string &prefix, DeviceCsr *merged,
                   const std::shared_ptr<DeviceCsr> &from_rules, const Tensor &rule_x,
                   const std::shared_ptr<DeviceCsr> &from_vertices, const Tensor &x) {
    const int64_t F = x.size(1);
    if (p.fuse_final && merged != nullptr) {
        Tensor out = torch::empty({merged->rows, F}, x.options());
        if (out.numel() == 0) return out;
        const int dtype = dtype_code(x);
        size_t bytes = 0;
        void *ws = nullptr;
        const std::shared_ptr<Scratch> scratch = merged->scratch;
        Hold hold(scratch->lock);
        cgnn_csr a = merged->prepare(F, dtype, p.kernel, &ws, &bytes);
        hipStream_t stream = reinterpret_cast<hipStream_t>(current_stream(x));
        const int id = p.timer.open(prefix + "final", stream);
        ok(cgnn_spmm_dual(&a, p.V, dtype, x.data_ptr(), rule_x.data_ptr(), out.data_ptr(), F, p.kernel, ws, bytes,
                          current_stream(x)),
           "spmm_dual");
        p.timer.close(id, stream);
        return out;
    }
    p.require_split_blocks();
    Tensor out = timed_spmm(p, prefix + "from_rules", *from_rules, rule_x, c10::nullopt);
    return timed_spmm(p, prefix + "from_vertices", *from_vertices, x, out);
}

// layer/CompressgnnSPMM.py:43-62 of the reference.  Stage names: fwd.rules (r2v),
// fwd.level<i>, fwd.final (v2r + v2v fused; alone where the rules are multiplied out) or fwd.from_rules / fwd.from_vertices.
Tensor propagate_forward(PropagationPlan &p, Tensor x) {
    require_gpu(x, "x");
    TORCH_CHECK(x.dim() == 2 && x.size(0) == p.V, "x must be [vertex_cnt, F]");
    x = x.contiguous();
    c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
    Hold hold(p.lock);
    if (auto whole = multiplied_out(p, p.whole, p.vertex_stage, p.r2v, x)) return timed_spmm(p, "fwd.final", *whole, x, c10::nullopt);
    Tensor rule_out = timed_spmm(p, "fwd.rules", *p.r2v, x, c10::nullopt);
    for (size_t i = 0; i < p.r2r.size(); ++i)
        rule_out = timed_spmm(p, "fwd.level" + std::to_string(i), *p.r2r[i], rule_out, rule_out);
    return final_stage(p, "fwd.", p.vertex_stage.get(), p.v2r, rule_out, p.v2v, x);
}

// A copy of a block that shares everything but the column numbers: the columns below
// `first_cols` go through `index` (cgnn_csr_compose_columns).
std::shared_ptr<DeviceCsr> compose_block(const DeviceCsr &A, const Tensor &narrow, int64_t first_cols, int64_t cols) {
    const std::shared_ptr<Scratch> scratch = A.scratch;
    Hold hold(scratch->lock);
    auto blk = std::make_shared<DeviceCsr>(A);
    blk->cols = cols;
    if (A.nnz > 0) {
        blk->colidx = torch::empty_like(A.colidx);
        ok(cgnn_csr_compose_columns(A.nnz, A.colidx.data_ptr<int32_t>(), first_cols, narrow.data_ptr<int32_t>(),
                                    blk->colidx.data_ptr<int32_t>(), current_stream(narrow)),
           "csr_compose_columns");
    }
    return blk;
}

// out = A * reps[index] over the compressed graph without reps[index]: the forward chain of
// propagate_forward on blocks whose vertex columns name the representative of the vertex.
// reps: [groups, F]; index: int64 [vertex_cnt] with values in [0, groups).  The same sums in the
// same order as propagate_forward(reps.index_select(0, index)): the same bits.  The composed
// blocks that the width takes are made on the first call for an index tensor (one host read: the ids are
// checked) and kept until that tensor is written to or freed.  Stage names: fwd.rules, fwd.level<i>, fwd.final.
Tensor propagate_forward_gathered(PropagationPlan &p, Tensor reps, Tensor index) {
    require_gpu(reps, "reps");
    require_gpu(index, "index");
    TORCH_CHECK(reps.dim() == 2 && reps.size(0) >= 1, "reps must be [groups, F] with at least one group");
    TORCH_CHECK(index.dim() == 1 && index.numel() == p.V && index.scalar_type() == torch::kInt64 && index.is_contiguous() &&
                    index.device() == reps.device(),
                "index must be a contiguous int64 tensor [vertex_cnt] on the device of reps");
    TORCH_CHECK(p.fused(), "propagation from representatives needs the fused vertex stage (plan.fuse_final = True)");
    reps = reps.contiguous();
    c10::hip::HIPGuardMasqueradingAsCUDA guard(reps.device());
    const int64_t groups = reps.size(0), F = reps.size(1);
    Hold hold(p.lock);
    const std::shared_ptr<DeviceCsr> whole = multiplied_out(p, p.whole, p.vertex_stage, p.r2v, reps);
    std::shared_ptr<PropagationPlan::Composed> known;
    for (auto it = p.composed.begin(); it != p.composed.end() && !known;) {
        if ((*it)->index.expired()) {
            it = p.composed.erase(it);
            continue;
        }
        if ((*it)->index._unsafe_get_target() == index.unsafeGetTensorImpl() && (*it)->version == index._version() &&
            (*it)->groups == groups)
            known = *it;
        ++it;
    }
    std::shared_ptr<DeviceCsr> rules, stage, composed_whole;
    if (known) rules = known->rules, stage = known->stage, composed_whole = known->whole;
    if (whole ? !composed_whole : !stage) {
        Tensor bad = torch::zeros({1}, index.options().dtype(torch::kInt32));
        Tensor narrow = torch::empty({p.V}, index.options().dtype(torch::kInt32));
        ok(cgnn_narrow_ids(p.V, index.data_ptr<int64_t>(), groups, narrow.data_ptr<int32_t>(), bad.data_ptr<int32_t>(),
                           current_stream(index)),
           "narrow_ids");
        if (whole) {
            composed_whole = compose_block(*whole, narrow, p.V, groups);
        } else {
            rules = compose_block(*p.r2v, narrow, p.V, groups);
            stage = compose_block(*p.vertex_stage, narrow, p.V, p.vertex_stage->cols);
        }
        if (known) {  // the ids were checked; what a capture makes is the graph's
            if (!capturing(index)) {
                TORCH_CHECK(synchronized(current_stream(index)), "propagate: the stream reported an error");
                known->rules = rules, known->stage = stage, known->whole = composed_whole;
            }
        } else {
            TORCH_CHECK(bad.item<int32_t>() == 0, "propagation from representatives: the index holds a cluster id outside [0, ", groups, ")");
        }
        if (!known && !index.is_inference()) {
            p.composed.push_front(std::make_shared<PropagationPlan::Composed>(PropagationPlan::Composed{
                c10::weak_intrusive_ptr<c10::TensorImpl>(index.getIntrusivePtr()), index._version(), groups, rules, stage, composed_whole}));
            while (p.composed.size() > 4) p.composed.pop_back();
        }
    }
    if (whole) return timed_spmm(p, "fwd.final", *composed_whole, reps, c10::nullopt);
    Tensor rule_out = timed_spmm(p, "fwd.rules", *rules, reps, c10::nullopt);
    for (size_t i = 0; i < p.r2r.size(); ++i)
        rule_out = timed_spmm(p, "fwd.level" + std::to_string(i), *p.r2r[i], rule_out, rule_out);
    Tensor out = torch::empty({p.V, F}, reps.options());
    if (out.numel() == 0) return out;
    const int dtype = dtype_code(reps);
    size_t bytes = 0;
    void *ws = nullptr;
    const std::shared_ptr<Scratch> scratch = stage->scratch;
    Hold products(scratch->lock);
    cgnn_csr a = stage->prepare(F, dtype, p.kernel, &ws, &bytes);
    hipStream_t stream = reinterpret_cast<hipStream_t>(current_stream(reps));
    const int id = p.timer.open("fwd.final", stream);
    ok(cgnn_spmm_dual(&a, p.V, dtype, reps.data_ptr(), rule_out.data_ptr(), out.data_ptr(), F, p.kernel, ws, bytes,
                      current_stream(reps)),
       "spmm_dual");
    p.timer.close(id, stream);
    return out;
}

// layer/CompressgnnSPMM.py:65-86 (the working branch, lines 80-85).  Stage names as in
// forward with the prefix bwd.
Tensor propagate_backward(PropagationPlan &p, Tensor grad) {
    require_gpu(grad, "grad");
    TORCH_CHECK(grad.dim() == 2 && grad.size(0) == p.V, "grad must be [vertex_cnt, F]");
    grad = grad.contiguous();
    c10::hip::HIPGuardMasqueradingAsCUDA guard(grad.device());
    Hold hold(p.lock);
    if (auto whole = multiplied_out(p, p.whole_t, p.vertex_stage_t, p.v2r_t, grad))
        return timed_spmm(p, "bwd.final", *whole, grad, c10::nullopt);
    Tensor rule_g = timed_spmm(p, "bwd.rules", *p.v2r_t, grad, c10::nullopt);
    for (size_t i = p.r2r_t.size(); i-- > 0;)
        rule_g = timed_spmm(p, "bwd.level" + std::to_string(i), *p.r2r_t[i], rule_g, rule_g);
    return final_stage(p, "bwd.", p.vertex_stage_t.get(), p.r2v_t, rule_g, p.v2v_t, grad);
}

// Where a native step of autograd does not do what an autograd function of Python does: under torch.jit.trace, which
// records a function as an operation on its inputs but the result of a native call as a constant; for inputs with a
// forward-mode tangent and under the transforms of torch.func, which a function without the rules for them refuses.
// There a native step does nothing and returns None, and the layer calls its function.
bool needs_function(const Tensor &a, const c10::optional<Tensor> &b = c10::nullopt) {
    return torch::jit::tracer::isTracing() || a._fw_grad(0).defined() || (b.has_value() && b->defined() && b->_fw_grad(0).defined()) ||
           c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode);
}

// A gradient asked for with create_graph, of a step that has first-order gradients only: it cannot be differentiated
// again and says so.
torch::autograd::variable_list first_order(torch::autograd::variable_list grads, bool recorded) {
    if (!recorded) return grads;
    auto refuse = std::make_shared<torch::autograd::DelayedError>(
        "trying to differentiate twice a function that has first-order gradients only (once_differentiable)", 1);
    for (Tensor &g : grads)
        if (g.defined()) g = (*refuse)({g.requires_grad() ? g : g.detach().requires_grad_()})[0];
    return grads;
}

// One propagation as a step of autograd.  The node is native, so a training step takes neither the
// interpreter nor its lock on the way back (the engine's thread and the caller's would pass the lock to each
// other): forward and gradient over 2,708 vertices took 69 us through a Python function and take 54 us so, 29
// of them the engine's own.
struct PropagateBackward : torch::autograd::Node {
    std::shared_ptr<PropagationPlan> plan;
    bool once = false;  // whether a second differentiation is refused (else the gradient counts as a constant there)
    torch::autograd::variable_list apply(torch::autograd::variable_list &&grads) override {
        if (!grads[0].defined()) return {Tensor()};
        const bool recorded = once && at::GradMode::is_enabled();
        Tensor out;
        {
            at::NoGradGuard no_grad;
            out = propagate_backward(*plan, grads[0]);
        }
        return first_order({out}, recorded);
    }
    std::string name() const override { return "PropagateBackward"; }
};

c10::optional<Tensor> propagate(const std::shared_ptr<PropagationPlan> &plan, const Tensor &x, bool once_differentiable) {
    if (needs_function(x)) return c10::nullopt;
    const bool differentiable = at::GradMode::is_enabled() && x.requires_grad();
    Tensor out;
    {
        at::NoGradGuard no_grad;
        out = propagate_forward(*plan, x);
    }
    if (differentiable) {
        std::shared_ptr<PropagateBackward> node(new PropagateBackward(), torch::autograd::deleteNode);
        node->plan = plan;
        node->once = once_differentiable;
        node->set_next_edges(torch::autograd::collect_next_edges(x));
        torch::autograd::set_history(out, node);
    }
    return out;
}

// ---------------------------------------------------- transformation compression ----

// Operand checks of the transformation-compression operators.  Every operator names its
// operands once, as a row of Operand records, and `expect` reports the first one that does not
// fit, saying what was asked for and what arrived.
enum class Role { Features, Ids, Counts, Bias };

struct Operand {
    Role role;
    const char *name;
    const Tensor *tensor;
};

std::string seen(const Tensor &t) {
    std::ostringstream os;
    os << t.scalar_type() << t.sizes() << " on " << t.device() << (t.is_contiguous() ? "" : ", not contiguous");
    return os.str();
}

// `anchor`: the operand whose device (and, for floating operands, precision) the others share.
void expect(const char *op, const Tensor &anchor, std::initializer_list<Operand> operands) {
    for (const Operand &o : operands) {
        const Tensor &t = *o.tensor;
        bool fits = t.defined() && t.is_cuda() && t.is_contiguous() && t.device() == anchor.device();
        const char *asked = "";
        switch (o.role) {
            case Role::Features:
                asked = "a contiguous [rows, width] float32 or float64 matrix on the GPU";
                fits = fits && t.dim() == 2 && (t.scalar_type() == torch::kFloat32 || t.scalar_type() == torch::kFloat64) &&
                       t.scalar_type() == anchor.scalar_type();
                break;
            case Role::Ids:
                asked = "a contiguous int64 vector of cluster ids beside the features";
                fits = fits && t.dim() == 1 && t.scalar_type() == torch::kInt64;
                break;
            case Role::Counts:
                asked = "a contiguous int32 vector with at least the empty cluster 0, beside the features";
                fits = fits && t.dim() == 1 && t.scalar_type() == torch::kInt32 && t.numel() > 0;
                break;
            case Role::Bias:
                asked = "a contiguous vector of the features' precision, beside the features";
                fits = fits && t.dim() == 1 && t.scalar_type() == anchor.scalar_type();
                break;
        }
        TORCH_CHECK(fits, op, ": ", o.name, " has to be ", asked, "; it is ", t.defined() ? seen(t) : "undefined");
    }
}

// Number of hash buckets for `bits` sign bits.
int64_t buckets_for(const char *op, int64_t bits) {
    TORCH_CHECK(0 <= bits && bits <= 30, op, ": between 0 and 30 hyperplanes are supported, ", bits, " asked for");
    return int64_t(1) << bits;
}

// The hyperplanes of an assignment: one column per sign bit, one row per input feature.
void expect_planes(const char *op, const Tensor &input, const Tensor &planes, int64_t bits) {
    expect(op, input, {{Role::Features, "input", &input}, {Role::Features, "hyperplanes", &planes}});
    TORCH_CHECK(planes.size(0) == input.size(1) && planes.size(1) == bits, op, ": ", bits, " hyperplanes over ",
                input.size(1), " features make a [", input.size(1), ", ", bits, "] matrix, not ", planes.sizes());
    TORCH_CHECK(input.size(0) < INT_MAX, op, ": ", input.size(0), " rows do not fit the int32 cluster sizes");
}

// cluster_workspace_cuda (src/runtime/csrc/cluster/cuda/cluster_kernel.cu:111-117):
// [bucket counts int32[2^bits], prefix int32[2^bits], scan scratch uint8[...]].
std::vector<Tensor> cluster_workspace(Tensor input, int64_t bits) {
    const char *op = "cluster_workspace";
    expect(op, input, {{Role::Features, "input", &input}});
    const int64_t buckets = buckets_for(op, bits);
    c10::hip::HIPGuardMasqueradingAsCUDA guard(input.device());
    auto ints = input.options().dtype(torch::kInt32);
    return {torch::empty({buckets}, ints), torch::empty({buckets}, ints),
            torch::empty({(int64_t)cgnn_lsh_scan_workspace_bytes((int)bits)}, input.options().dtype(torch::kUInt8))};
}

// Assignment and member lists of one refresh: ids [N] int64 (1-based), counts
// [active+1] int32 (entry 0 = 0), active, and the member lists (offsets [active+2], perm
// [N], sorted_id [N], and a host scalar with the size of the largest group).  The codes are grouped by a stable sort instead of bucket counters,
// so the result is the same as cluster_assign_cuda's (cluster_kernel.cu:118-153) whatever
// the distribution of the codes, and the member lists come with it.  The number of groups
// is at most min(N, 2^bits): every kernel runs on buffers of that bound, so the device
// never waits for the host; the one scalar read of a refresh (cluster_kernel.cu:146-147)
// comes last and only trims the views.
int64_t largest_group(const std::vector<Tensor> &m) { return m.size() == 4 ? m[3].item<int64_t>() : 0; }

// Waits until a word of pinned memory is no longer `not_yet`.  The last thing that a launch writes is there while what
// stands behind it still runs: look for it as long as `patience`, and otherwise wait for the stream, which also reports its
// errors.  After kShortWait the interpreter's other threads may run.  (Not before: a thread that lets go of the lock has it back
// when the one that took it gives it up, after 5 ms if that one computes.)
constexpr std::chrono::microseconds kShortWait(200);

void await(const int32_t *word, int32_t not_yet, std::chrono::microseconds patience, cgnn_stream_t stream, const char *op) {
    const auto begin = std::chrono::steady_clock::now();
    auto arrives_within = [&](std::chrono::microseconds wait) {
        while (__atomic_load_n(word, __ATOMIC_ACQUIRE) == not_yet)
            if (std::chrono::steady_clock::now() - begin > wait) return false;
        return true;
    };
    if (arrives_within(std::min(patience, kShortWait))) return;
    std::optional<pybind11::gil_scoped_release> others;
    if (PyGILState_Check()) others.emplace();
    if (patience > kShortWait && arrives_within(patience)) return;
    TORCH_CHECK(hipStreamSynchronize(reinterpret_cast<hipStream_t>(stream)) == hipSuccess, op, ": the stream reported an error");
    TORCH_CHECK(__atomic_load_n(word, __ATOMIC_ACQUIRE) != not_yet, op, ": the sizes were not written");
}

struct Assigned {
    Tensor ids, counts, reps;
    int64_t active = 0;
    std::vector<Tensor> members;
};

// with_reps: the means of the rows over the clusters as well, launched before the host read where the buffer
// for all clusters there could be is small (kSmallReps elements; the rows behind the last cluster stay unused) and
// no cluster can be so large that its size, which is not known yet, would change how it is summed.
constexpr int64_t kSmallReps = int64_t(1) << 22;
constexpr int64_t kSmallClusters = int64_t(1) << 16;

Tensor member_means(const char *op, const Tensor &rows, const Tensor *counts, const std::vector<Tensor> &m, int64_t groups,
                    int64_t largest);

Assigned assign(Tensor input, Tensor planes, int64_t bits, bool with_reps) {
    const char *op = "cluster_assign";
    const int64_t buckets = buckets_for(op, bits);
    expect_planes(op, input, planes, bits);
    c10::hip::HIPGuardMasqueradingAsCUDA guard(input.device());
    const int64_t N = input.size(0), F = input.size(1);
    auto ints = input.options().dtype(torch::kInt32);
    Assigned a;
    a.ids = torch::empty({N}, input.options().dtype(torch::kInt64));
    auto host_scalar = [](int64_t v) { return torch::full({1}, v, torch::TensorOptions().dtype(torch::kInt64)); };
    if (N == 0) {
        a.counts = torch::zeros({1}, ints);
        a.members = {torch::zeros({2}, ints), torch::empty({0}, ints), torch::empty({0}, ints), host_scalar(0)};
        if (with_reps) a.reps = torch::zeros({1, F}, input.options());
        return a;
    }
    const int64_t cap = std::min<int64_t>(N, buckets);
    // each on its own: with the three in one buffer the spread over perm took 512 us for 484 at 2.4 M x 256
    Tensor perm = torch::empty({N}, ints), sorted_id = torch::empty({N}, ints), codes = torch::empty({N}, ints);
    int32_t *raw = codes.data_ptr<int32_t>();
    Tensor sizes = torch::empty({2 * cap + 3}, ints);
    Tensor offsets = sizes.narrow(0, 0, cap + 2), counts = sizes.narrow(0, cap + 2, cap + 1);
    // number of groups, largest group: the grouping writes them with plain stores, on the host at once
    Tensor summary = torch::empty({2}, torch::TensorOptions().dtype(torch::kInt32).pinned_memory(true));
    constexpr int32_t kNotYet = -1;
    __atomic_store_n(summary.data_ptr<int32_t>(), kNotYet, __ATOMIC_RELAXED);
    auto stream = current_stream(input);
    // The pool of pinned memory knows nothing of the launch that writes `summary`: an error before the host read (no
    // room for the representatives) waits for it.
    struct Settle {
        hipStream_t stream;
        bool pending = false;
        ~Settle() {
            if (pending) (void)hipStreamSynchronize(stream);
        }
    } settle{reinterpret_cast<hipStream_t>(stream)};
    ok(cgnn_lsh_hash(N, F, (int)bits, dtype_code(input), input.data_ptr(), planes.data_ptr(), raw, nullptr, stream), "lsh_hash");
    const size_t bytes = cgnn_lsh_group_workspace_bytes(N, (int)bits);
    Tensor ws = torch::empty({(int64_t)std::max<size_t>(bytes, 1)}, input.options().dtype(torch::kUInt8));
    settle.pending = true;
    ok(cgnn_lsh_group(N, (int)bits, raw, a.ids.data_ptr<int64_t>(), offsets.data_ptr<int32_t>(), perm.data_ptr<int32_t>(),
                      sorted_id.data_ptr<int32_t>(), counts.data_ptr<int32_t>(), summary.data_ptr<int32_t>(), ws.data_ptr(), bytes,
                      stream),
       "lsh_group");
    const std::vector<Tensor> wide_lists = {offsets, perm, sorted_id};
    const bool early = with_reps && F > 0 && (cap + 1) * F <= kSmallReps && N <= kSmallClusters;
    if (early) a.reps = member_means("cluster_mean", input, nullptr, wide_lists, cap + 1, N);
    // The one host read of a refresh, in a stream with a training step ahead.  A copy behind the launch takes the host
    // 24 us, a refresh of 60,000 rows and its products 262 us with it and 220 so; waiting for the stream after 200 us already
    // makes a step of 3.77 ms 20 us longer.
    await(summary.data_ptr<int32_t>(), kNotYet, std::chrono::milliseconds(5), stream, op);
    settle.pending = false;
    a.active = summary.data_ptr<int32_t>()[0];
    a.counts = counts.narrow(0, 0, a.active + 1);
    a.members = {offsets.narrow(0, 0, a.active + 2), perm, sorted_id, host_scalar(summary.data_ptr<int32_t>()[1])};
    if (early) a.reps = a.reps.narrow(0, 0, a.active + 1);
    else if (with_reps && F > 0) a.reps = member_means("cluster_mean", input, nullptr, a.members, a.active + 1, largest_group(a.members));
    else if (with_reps) a.reps = torch::zeros({a.active + 1, F}, input.options());
    return a;
}

std::tuple<Tensor, Tensor, int64_t, std::vector<Tensor>> cluster_assign_members(Tensor input, Tensor planes, int64_t bits) {
    Assigned a = assign(input, planes, bits, false);
    return {a.ids, a.counts, a.active, a.members};
}

// Member lists by the index tensor they belong to.  The operators with the reference's
// signatures (cluster_mean(input, index, count), cluster_reconstruct(reps, index, bias, relu), ...)
// receive an index and nothing else; the lists that go with it, and the knowledge that its ids
// were checked, are kept here so that only the first call on an index builds them (one host
// read), as the reference reads the host once per assignment (cluster_kernel.cu:147).  An entry
// names its tensor by a weak reference and the tensor's version counter: it is dropped when the
// tensor is freed and ignored once the tensor was written to.
struct MemberCache {
    struct Entry {
        c10::weak_intrusive_ptr<c10::TensorImpl> index;
        uint32_t version;
        int64_t groups;
        std::vector<Tensor> members;
    };
    static constexpr size_t kKeep = 8;
    std::deque<Entry> entries;
    std::mutex lock;

    bool find(const Tensor &index, int64_t groups, std::vector<Tensor> *out) {
        std::lock_guard<std::mutex> hold(lock);
        for (auto it = entries.begin(); it != entries.end();) {
            if (it->index.expired()) {
                it = entries.erase(it);
                continue;
            }
            if (it->index._unsafe_get_target() == index.unsafeGetTensorImpl() && it->version == index._version() &&
                (groups < 0 || it->groups == groups)) {
                *out = it->members;
                return true;
            }
            ++it;
        }
        return false;
    }
    void put(const Tensor &index, int64_t groups, std::vector<Tensor> members) {
        if (index.is_inference()) return;  // no version counter to tell a later write by
        std::lock_guard<std::mutex> hold(lock);
        entries.push_front(Entry{c10::weak_intrusive_ptr<c10::TensorImpl>(index.getIntrusivePtr()), index._version(),
                                 groups, std::move(members)});
        while (entries.size() > kKeep) entries.pop_back();
    }
};

MemberCache &member_cache() {
    static MemberCache cache;
    return cache;
}

// cluster_assign_cuda (cluster_kernel.cu:118-153).  The three tensors of cluster_workspace
// are accepted, and must be what cluster_workspace returns for these arguments; the grouping
// itself sorts the codes and no longer touches bucket counters.
std::tuple<Tensor, Tensor, int64_t> cluster_assign(Tensor input, Tensor planes, int64_t bits,
                                                   std::vector<Tensor> workspace) {
    const char *op = "cluster_assign";
    const int64_t buckets = buckets_for(op, bits);
    expect_planes(op, input, planes, bits);
    TORCH_CHECK(workspace.size() == 3, op, ": the workspace is the three tensors of cluster_workspace, ", workspace.size(),
                " given");
    const int64_t need[3] = {buckets, buckets, (int64_t)cgnn_lsh_scan_workspace_bytes((int)bits)};
    const torch::ScalarType kind[3] = {torch::kInt32, torch::kInt32, torch::kUInt8};
    for (int i = 0; i < 3; ++i) {
        const Tensor &w = workspace[i];
        const bool fits = w.defined() && w.device() == input.device() && w.dim() == 1 && w.is_contiguous() &&
                          w.scalar_type() == kind[i] && (i < 2 ? w.numel() == need[i] : w.numel() >= need[i]);
        TORCH_CHECK(fits, op, ": workspace[", i, "] has to be ", kind[i], "[", need[i], "] beside the input; it is ",
                    w.defined() ? seen(w) : "undefined");
    }
    auto grouped = cluster_assign_members(input, planes, bits);
    // the lists made along the way stay with the ids: the operators that are handed these ids
    // (and nothing else) find them again
    member_cache().put(std::get<0>(grouped), std::get<2>(grouped) + 1, std::get<3>(grouped));
    return {std::get<0>(grouped), std::get<1>(grouped), std::get<2>(grouped)};
}

// cluster_forward (src/runtime/csrc/cluster/cluster.cpp:12-30): int32 ids and the
// number of active buckets.
std::tuple<Tensor, int64_t> cluster_forward(Tensor input, Tensor random_vectors, int64_t param_h) {
    require_gpu(input, "input");
    auto grouped = cluster_assign_members(input, random_vectors, param_h);
    return {std::get<0>(grouped).to(torch::kInt32), std::get<2>(grouped)};
}

// One int32 on the device that the kernels set when they meet a cluster id that names no
// cluster; `raise` reads it (the only host read of these operators, made only for index
// tensors that do not come with member lists of this library's own making).
struct IdFlag {
    Tensor flag;
    explicit IdFlag(const Tensor &like) : flag(torch::zeros({1}, like.options().dtype(torch::kInt32))) {}
    int32_t *ptr() { return flag.data_ptr<int32_t>(); }
    void raise(const char *op, int64_t groups) {
        TORCH_CHECK(flag.item<int32_t>() == 0, op, ": the index holds a cluster id outside [0, ", groups, ")");
    }
};

// Member lists of `groups` clusters: [offsets int32[groups+1], perm int32[N], sorted_id int32[N]].
std::vector<Tensor> cluster_members(Tensor index, int64_t groups) {
    const char *op = "cluster_members";
    require_gpu(index, "index");
    expect(op, index, {{Role::Ids, "index", &index}});
    TORCH_CHECK(groups >= 1, op, ": at least the empty cluster 0 is needed, groups = ", groups);
    c10::hip::HIPGuardMasqueradingAsCUDA guard(index.device());
    const int64_t N = index.numel();
    auto i32 = index.options().dtype(torch::kInt32);
    Tensor offsets = torch::empty({groups + 1}, i32), perm = torch::empty({N}, i32), sorted = torch::empty({N}, i32);
    const size_t bytes = cgnn_cluster_members_workspace_bytes(N, groups);
    Tensor ws = torch::empty({(int64_t)std::max<size_t>(bytes, 1)}, index.options().dtype(torch::kUInt8));
    IdFlag bad(index);
    ok(cgnn_cluster_members(N, groups, N ? index.data_ptr<int64_t>() : nullptr, offsets.data_ptr<int32_t>(),
                            N ? perm.data_ptr<int32_t>() : nullptr, N ? sorted.data_ptr<int32_t>() : nullptr, bad.ptr(),
                            ws.data_ptr(), bytes, current_stream(index)),
       op);
    bad.raise(op, groups);
    return {offsets, perm, sorted};
}

// Member lists handed in by the caller ([offsets, perm, sorted_id] and optionally a host int64
// scalar with the size of the largest group), checked against the index they belong to.
bool has_members(const c10::optional<std::vector<Tensor>> &members) { return members.has_value() && !members->empty(); }

void expect_members(const char *op, const std::vector<Tensor> &m, const Tensor &index, int64_t groups) {
    TORCH_CHECK(m.size() == 3 || m.size() == 4, op, ": member lists are [offsets, perm, sorted_id] (+ largest group), ",
                m.size(), " tensors given");
    const int64_t want[3] = {groups + 1, index.numel(), index.numel()};
    const char *names[3] = {"offsets", "perm", "sorted_id"};
    for (int i = 0; i < 3; ++i)
        TORCH_CHECK(m[i].defined() && m[i].scalar_type() == torch::kInt32 && m[i].device() == index.device() &&
                        m[i].is_contiguous() && (groups < 0 && i == 0 ? true : m[i].numel() == want[i]),
                    op, ": member list '", names[i], "' has to be int32[", want[i], "] beside the index; it is ",
                    m[i].defined() ? seen(m[i]) : "undefined");
    if (m.size() == 4)
        TORCH_CHECK(!m[3].is_cuda() && m[3].numel() == 1 && m[3].scalar_type() == torch::kInt64, op,
                    ": the fourth member tensor is a host int64 scalar (size of the largest group)");
}

std::vector<Tensor> members_or_build(const char *op, const c10::optional<std::vector<Tensor>> &members,
                                     const Tensor &index, int64_t groups) {
    if (has_members(members)) {
        expect_members(op, *members, index, groups);
        return *members;
    }
    std::vector<Tensor> known;
    if (member_cache().find(index, groups, &known)) return known;
    known = cluster_members(index, groups);  // checks the ids: the one host read for this index
    member_cache().put(index, groups, known);
    return known;
}

// Sums over the members of every group, [groups, F]; rows has at least one element.  mask as in cgnn_cluster_sums.
Tensor member_sums(const char *op, const Tensor &rows, int mask, const void *M, const std::vector<Tensor> &m, int64_t groups) {
    const int64_t N = rows.size(0), F = rows.size(1);
    const int dtype = dtype_code(rows);
    const int32_t *offsets = m[0].data_ptr<int32_t>(), *perm = m[1].data_ptr<int32_t>(), *sorted_id = m[2].data_ptr<int32_t>();
    const auto stream = current_stream(rows);
    Tensor out = torch::empty({groups, F}, rows.options());
    int64_t arrivals = 0;
    size_t bytes = cgnn_cluster_sums_workspace_bytes(N, F, groups, dtype, &arrivals);
    if (arrivals == 0) bytes = cgnn_cluster_mean_workspace_bytes(N, F, groups, dtype);
    Tensor ws = torch::empty({(int64_t)std::max<size_t>(bytes, 1)}, rows.options().dtype(torch::kUInt8));
    if (arrivals > 0) {
        Tensor counters = arrival_pool().get(arrivals, rows);
        ok(cgnn_cluster_sums(N, F, groups, dtype, rows.data_ptr(), mask, M, offsets, perm, sorted_id, out.data_ptr(), ws.data_ptr(),
                             bytes, counters.data_ptr<int32_t>(), stream),
           op);
    } else if (mask >= 2) {
        const auto run = mask == 3 ? cgnn_reconstruct_backward_masks : cgnn_reconstruct_backward_signs;
        ok(run(N, F, groups, largest_group(m), dtype, rows.data_ptr(), static_cast<const uint32_t *>(M), offsets, perm, sorted_id,
               out.data_ptr(), ws.data_ptr(), bytes, stream),
           op);
    } else {
        ok(cgnn_reconstruct_backward(N, F, groups, largest_group(m), dtype, rows.data_ptr(), M, offsets, perm, sorted_id, mask,
                                     out.data_ptr(), ws.data_ptr(), bytes, stream),
           op);
    }
    return out;
}

// Means over the members of every group: by the caller's counts, or (NULL) by the lengths of the lists.
// largest: the size of the largest group or a bound on it, 0 if unknown.
Tensor member_means(const char *op, const Tensor &rows, const Tensor *counts, const std::vector<Tensor> &m, int64_t groups,
                    int64_t largest) {
    const int64_t N = rows.size(0), F = rows.size(1);
    const int dtype = dtype_code(rows);
    Tensor out = torch::empty({groups, F}, rows.options());
    const size_t bytes = cgnn_cluster_mean_workspace_bytes(N, F, groups, dtype);
    Tensor ws = torch::empty({(int64_t)std::max<size_t>(bytes, 1)}, rows.options().dtype(torch::kUInt8));
    ok(cgnn_cluster_mean(N, F, groups, largest, dtype, rows.data_ptr(), m[0].data_ptr<int32_t>(), m[1].data_ptr<int32_t>(),
                         m[2].data_ptr<int32_t>(), counts ? counts->data_ptr<int32_t>() : nullptr, out.data_ptr(),
                         ws.data_ptr(), bytes, current_stream(rows)),
       op);
    return out;
}

// cluster_mean_cuda (cluster_kernel.cu:158-170).  `members` (from cluster_members, for
// the same index) avoids rebuilding the member lists on every call.
Tensor cluster_mean(Tensor input, Tensor index, Tensor count, c10::optional<std::vector<Tensor>> members) {
    const char *op = "cluster_mean";
    expect(op, input, {{Role::Features, "input", &input}, {Role::Ids, "index", &index}, {Role::Counts, "count", &count}});
    TORCH_CHECK(index.numel() == input.size(0), op, ": ", input.size(0), " rows but ", index.numel(), " cluster ids");
    c10::hip::HIPGuardMasqueradingAsCUDA guard(input.device());
    const int64_t groups = count.numel();
    if (input.numel() == 0) return torch::zeros({groups, input.size(1)}, input.options());
    auto m = members_or_build(op, members, index, groups);
    return member_means(op, input, &count, m, groups, largest_group(m));  // the counts need not be the lists' lengths
}

// The order in which a gather produces its rows: the member list `perm` when the caller has one
// or an earlier operator on the same index has left one (`held` keeps it alive for the call).
// An index met for the first time, without lists, is an index from outside the assignment
// operators: its ids are checked by the gather itself (one host read) and its lists are built
// for the calls that follow.
const int32_t *production_order(const char *op, const c10::optional<std::vector<Tensor>> &members, const Tensor &index,
                                int64_t groups, std::vector<Tensor> *held) {
    if (has_members(members)) {
        expect_members(op, *members, index, -1);
        return (*members)[1].data_ptr<int32_t>();
    }
    if (member_cache().find(index, groups, held)) return (*held)[1].data_ptr<int32_t>();
    return nullptr;
}

// After a gather over an index that had no lists: the flag is read (the ids are then known to be
// good) and the lists are made, so that later operators on this index read nothing.
void remember_checked_index(const char *op, IdFlag &bad, const Tensor &index, int64_t groups) {
    bad.raise(op, groups);
    if (groups >= 1) member_cache().put(index, groups, cluster_members(index, groups));
}

// cluster_mean_backward_cuda (cluster_kernel.cu:171-181).
Tensor cluster_mean_backward(Tensor grad, Tensor index, Tensor count, c10::optional<std::vector<Tensor>> members) {
    const char *op = "cluster_mean_backward";
    expect(op, grad, {{Role::Features, "grad", &grad}, {Role::Ids, "index", &index}, {Role::Counts, "count", &count}});
    TORCH_CHECK(grad.size(0) == count.numel(), op, ": ", grad.size(0), " gradient rows for ", count.numel(), " clusters");
    c10::hip::HIPGuardMasqueradingAsCUDA guard(grad.device());
    Tensor out = torch::empty({index.numel(), grad.size(1)}, grad.options());
    if (out.numel() == 0) return out;
    std::vector<Tensor> held;
    const int32_t *perm = production_order(op, members, index, count.numel(), &held);
    c10::optional<IdFlag> bad;
    if (perm == nullptr) bad.emplace(index);
    ok(cgnn_cluster_mean_backward(index.numel(), grad.size(1), count.numel(), dtype_code(grad), grad.data_ptr(),
                                  index.data_ptr<int64_t>(), count.data_ptr<int32_t>(), perm, out.data_ptr(),
                                  bad ? bad->ptr() : nullptr, current_stream(grad)),
       op);
    if (bad) remember_checked_index(op, *bad, index, count.numel());
    return out;
}

// cluster_reconstruct_cuda (cluster_kernel.cu:182-195).
Tensor cluster_reconstruct(Tensor reps, Tensor index, c10::optional<Tensor> bias, bool relu,
                           c10::optional<std::vector<Tensor>> members) {
    const char *op = "cluster_reconstruct";
    expect(op, reps, {{Role::Features, "representatives", &reps}, {Role::Ids, "index", &index}});
    if (bias.has_value()) {
        expect(op, reps, {{Role::Bias, "bias", &*bias}});
        TORCH_CHECK(bias->numel() == reps.size(1), op, ": a bias of ", bias->numel(), " entries for rows of ", reps.size(1));
    }
    TORCH_CHECK(index.numel() == 0 || reps.size(0) > 0, op, ": rows to reconstruct but no representatives");
    c10::hip::HIPGuardMasqueradingAsCUDA guard(reps.device());
    Tensor out = torch::empty({index.numel(), reps.size(1)}, reps.options());
    if (out.numel() == 0) return out;
    std::vector<Tensor> held;
    const int32_t *perm = production_order(op, members, index, reps.size(0), &held);
    c10::optional<IdFlag> bad;
    if (perm == nullptr) bad.emplace(index);
    ok(cgnn_reconstruct(index.numel(), reps.size(1), reps.size(0), dtype_code(reps), reps.data_ptr(),
                        index.data_ptr<int64_t>(), perm, bias.has_value() ? bias->data_ptr() : nullptr, relu ? 1 : 0,
                        out.data_ptr(), bad ? bad->ptr() : nullptr, current_stream(reps)),
       op);
    if (bad) remember_checked_index(op, *bad, index, reps.size(0));
    return out;
}

// cluster_reconstruct_backward_cuda (cluster_kernel.cu:196-208).
Tensor cluster_reconstruct_backward(Tensor grad, Tensor index, Tensor output, int64_t groups, bool relu,
                                    c10::optional<std::vector<Tensor>> members) {
    const char *op = "cluster_reconstruct_backward";
    expect(op, grad, {{Role::Features, "grad", &grad}, {Role::Ids, "index", &index}, {Role::Features, "output", &output}});
    TORCH_CHECK(groups >= 0, op, ": groups = ", groups);
    TORCH_CHECK(output.sizes() == grad.sizes(), op, ": the saved output is ", output.sizes(), ", the gradient ", grad.sizes());
    TORCH_CHECK(index.numel() == grad.size(0), op, ": ", grad.size(0), " rows but ", index.numel(), " cluster ids");
    c10::hip::HIPGuardMasqueradingAsCUDA guard(grad.device());
    const int64_t N = grad.size(0), F = grad.size(1);
    if (grad.numel() == 0 || groups == 0) return torch::zeros({groups, F}, grad.options());
    auto m = members_or_build(op, members, index, groups);
    return member_sums(op, grad, relu ? 1 : 0, relu ? output.data_ptr() : nullptr, m, groups);
}

// The ReLU form of cluster_reconstruct that also returns the sign of every output element as one
// bit: (rows [N, F], signs int32 [N, ceil(F / 32)]), or, by group, masks int32 [groups, ceil(F / 32)]: the rows
// of a group are copies of one representative and have the same signs.  Words of groups that do not occur are not written.
std::tuple<Tensor, Tensor> reconstruct_with_signs(const char *op, const Tensor &reps, const Tensor &index,
                                                  const c10::optional<Tensor> &bias, const c10::optional<std::vector<Tensor>> &members,
                                                  bool by_group) {
    expect(op, reps, {{Role::Features, "representatives", &reps}, {Role::Ids, "index", &index}});
    if (bias.has_value()) {
        expect(op, reps, {{Role::Bias, "bias", &*bias}});
        TORCH_CHECK(bias->numel() == reps.size(1), op, ": a bias of ", bias->numel(), " entries for rows of ", reps.size(1));
    }
    TORCH_CHECK(index.numel() == 0 || reps.size(0) > 0, op, ": rows to reconstruct but no representatives");
    c10::hip::HIPGuardMasqueradingAsCUDA guard(reps.device());
    const int64_t N = index.numel(), F = reps.size(1);
    Tensor out = torch::empty({N, F}, reps.options());
    Tensor signs = torch::empty({by_group ? reps.size(0) : N, cgnn_sign_words(F)}, reps.options().dtype(torch::kInt32));
    if (out.numel() == 0) return {out, signs};
    std::vector<Tensor> held;
    const int32_t *perm = production_order(op, members, index, reps.size(0), &held);
    c10::optional<IdFlag> bad;
    if (perm == nullptr) bad.emplace(index);
    const auto run = by_group ? cgnn_reconstruct_masks : cgnn_reconstruct_signs;
    ok(run(N, F, reps.size(0), dtype_code(reps), reps.data_ptr(), index.data_ptr<int64_t>(), perm,
           bias.has_value() ? bias->data_ptr() : nullptr, out.data_ptr(), reinterpret_cast<uint32_t *>(signs.data_ptr<int32_t>()),
           bad ? bad->ptr() : nullptr, current_stream(reps)),
       op);
    if (bad) remember_checked_index(op, *bad, index, reps.size(0));
    return {out, signs};
}

// cluster_reconstruct_backward with relu = true, the mask taken from the words above.
Tensor reconstruct_backward_with_signs(const char *op, const Tensor &grad, const Tensor &index, const Tensor &signs, int64_t groups,
                                       const c10::optional<std::vector<Tensor>> &members, bool by_group) {
    expect(op, grad, {{Role::Features, "grad", &grad}, {Role::Ids, "index", &index}});
    TORCH_CHECK(groups >= 0, op, ": groups = ", groups);
    TORCH_CHECK(index.numel() == grad.size(0), op, ": ", grad.size(0), " rows but ", index.numel(), " cluster ids");
    const int64_t N = grad.size(0), F = grad.size(1), of = by_group ? groups : N;
    TORCH_CHECK(signs.device() == grad.device() && signs.scalar_type() == torch::kInt32 && signs.is_contiguous() &&
                    signs.dim() == 2 && signs.size(0) == of && signs.size(1) == cgnn_sign_words(F),
                op, by_group ? ": masks" : ": signs", " must be a contiguous int32 tensor [", of, ", ", cgnn_sign_words(F),
                "] on the device of grad");
    c10::hip::HIPGuardMasqueradingAsCUDA guard(grad.device());
    if (grad.numel() == 0 || groups == 0) return torch::zeros({groups, F}, grad.options());
    auto m = members_or_build(op, members, index, groups);
    return member_sums(op, grad, by_group ? 3 : 2, signs.data_ptr<int32_t>(), m, groups);
}

std::tuple<Tensor, Tensor> cluster_reconstruct_signs(Tensor reps, Tensor index, c10::optional<Tensor> bias,
                                                     c10::optional<std::vector<Tensor>> members) {
    return reconstruct_with_signs("cluster_reconstruct_signs", reps, index, bias, members, false);
}

Tensor cluster_reconstruct_backward_signs(Tensor grad, Tensor index, Tensor signs, int64_t groups,
                                          c10::optional<std::vector<Tensor>> members) {
    return reconstruct_backward_with_signs("cluster_reconstruct_backward_signs", grad, index, signs, groups, members, false);
}

// By group: what a layer may keep for its backward pass (the reference keeps the rows: layer/CompressgnnReconstruct.py:16-22).
std::tuple<Tensor, Tensor> cluster_reconstruct_masks(Tensor reps, Tensor index, c10::optional<Tensor> bias,
                                                     c10::optional<std::vector<Tensor>> members) {
    return reconstruct_with_signs("cluster_reconstruct_masks", reps, index, bias, members, true);
}

Tensor cluster_reconstruct_backward_masks(Tensor grad, Tensor index, Tensor masks, int64_t groups,
                                          c10::optional<std::vector<Tensor>> members) {
    return reconstruct_backward_with_signs("cluster_reconstruct_backward_masks", grad, index, masks, groups, members, true);
}

// ------------------------------------------------------ the layers' autograd steps ----
//
// Native nodes, for the reason given at PropagateBackward.  They give first-order gradients, as the reference's
// functions do.

template <typename Node>
std::shared_ptr<Node> node_over(const Tensor &a, const Tensor &b = Tensor()) {
    std::shared_ptr<Node> node(new Node(), torch::autograd::deleteNode);
    node->set_next_edges(b.defined() ? torch::autograd::collect_next_edges(a, b) : torch::autograd::collect_next_edges(a));
    return node;
}

using Members = c10::optional<std::vector<Tensor>>;

struct MeanBackward : torch::autograd::Node {
    torch::autograd::SavedVariable index, counts;
    Members members;
    torch::autograd::variable_list apply(torch::autograd::variable_list &&grads) override {
        if (!grads[0].defined()) return {Tensor()};
        const bool recorded = at::GradMode::is_enabled();
        Tensor out;
        {
            at::NoGradGuard no_grad;
            out = cluster_mean_backward(grads[0].contiguous(), index.unpack(), counts.unpack(), members);
        }
        return first_order({out}, recorded);
    }
    void release_variables() override {
        index.reset_data();
        counts.reset_data();
        members.reset();
    }
    std::string name() const override { return "ClusterMeanBackward"; }
};

void attach_mean(Tensor &reps, const Tensor &x, const Tensor &index, const Tensor &counts, const Members &members) {
    if (!at::GradMode::is_enabled() || !x.requires_grad()) return;
    auto node = node_over<MeanBackward>(x);
    node->index = torch::autograd::SavedVariable(index, false);
    node->counts = torch::autograd::SavedVariable(counts, false);
    node->members = members;
    torch::autograd::set_history(reps, node);
}

// Representatives of an assignment that is held: the means of x over its clusters (the counts are the
// lengths of its lists).
c10::optional<Tensor> cluster_representatives(Tensor x, Tensor index, Tensor counts, std::vector<Tensor> members) {
    const char *op = "cluster_mean";
    if (needs_function(x)) return c10::nullopt;
    Tensor reps;
    {
        at::AutoDispatchBelowADInplaceOrView plain;
        Tensor rows = x.contiguous();
        expect(op, rows, {{Role::Features, "input", &rows}, {Role::Ids, "index", &index}, {Role::Counts, "count", &counts}});
        TORCH_CHECK(index.numel() == rows.size(0), op, ": ", rows.size(0), " rows but ", index.numel(), " cluster ids");
        expect_members(op, members, index, counts.numel());
        c10::hip::HIPGuardMasqueradingAsCUDA guard(rows.device());
        reps = rows.numel() == 0 ? torch::zeros({counts.numel(), rows.size(1)}, rows.options())
                                 : member_means(op, rows, nullptr, members, counts.numel(), largest_group(members));
    }
    attach_mean(reps, x, index, counts, members);
    return reps;
}

// A refresh: (representatives, ids, counts, active, member lists).
c10::optional<std::tuple<Tensor, Tensor, Tensor, int64_t, std::vector<Tensor>>> cluster_refresh(Tensor x, Tensor planes,
                                                                                              int64_t bits) {
    if (needs_function(x)) return c10::nullopt;
    Assigned a;
    {
        at::AutoDispatchBelowADInplaceOrView plain;
        a = assign(x.contiguous(), planes.contiguous(), bits, true);
    }
    attach_mean(a.reps, x, a.ids, a.counts, a.members);
    return std::make_tuple(a.reps, a.ids, a.counts, a.active, a.members);
}

// Column sums of a [rows, F] matrix: the gradient of a bias.
Tensor column_sums(const Tensor &x) {
    const char *op = "column_sums";
    expect(op, x, {{Role::Features, "x", &x}});
    const int64_t rows = x.size(0), F = x.size(1);
    if (x.numel() == 0) return torch::zeros({F}, x.options());
    c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
    Tensor out = torch::empty({F}, x.options());
    int64_t arrivals = 0;
    const size_t bytes = cgnn_column_sums_workspace_bytes(rows, F, dtype_code(x), &arrivals);
    Tensor ws = torch::empty({(int64_t)std::max<size_t>(bytes, 1)}, x.options().dtype(torch::kUInt8));
    Tensor counters = arrival_pool().get(arrivals, x);
    ok(cgnn_column_sums(rows, F, dtype_code(x), x.data_ptr(), out.data_ptr(), ws.data_ptr(), bytes, counters.data_ptr<int32_t>(),
                        current_stream(x)),
       op);
    return out;
}

struct ReconstructBackward : torch::autograd::Node {
    torch::autograd::SavedVariable index, signs;  // signs: one bit per element, where the rows went through a ReLU
    Members members;
    int64_t groups = 0;
    bool relu = false, by_group = false, with_bias = false;  // by_group: bits of the representatives, not of the rows
    torch::autograd::variable_list apply(torch::autograd::variable_list &&grads) override {
        const size_t inputs = with_bias ? 2 : 1;
        if (!grads[0].defined()) return torch::autograd::variable_list(inputs);
        const bool recorded = at::GradMode::is_enabled();
        torch::autograd::variable_list out;
        {
            at::NoGradGuard no_grad;
            const Tensor d_rows = grads[0].contiguous(), ids = index.unpack();
            // without a ReLU the operator does not read the rows it is given as output
            out.push_back(relu ? reconstruct_backward_with_signs("cluster_reconstruct backward", d_rows, ids, signs.unpack(), groups,
                                                                 members, by_group)
                               : cluster_reconstruct_backward(d_rows, ids, d_rows, groups, false, members));
            if (with_bias) out.push_back(task_should_compute_output(1) ? column_sums(out[0]) : Tensor());
        }
        return first_order(std::move(out), recorded);
    }
    void release_variables() override {
        index.reset_data();
        signs.reset_data();
        members.reset();
    }
    std::string name() const override { return "ReconstructBackward"; }
};

// Whether a layer keeps the bits of the representatives or those of the rows.  The former save a cache line a member where the
// rows are summed, and all but a row of words per representative of what is held until then (1.3 of 78 MB for 2,449,029 rows of 256
// features); where rows that follow each other belong to different representatives their words are stored one by one, which costs most
// where a row ends inside a word.  So they are kept for many rows a representative, or few where a row is one word or whole ones.  (us,
// a forward and its gradient, bits of the rows / of the representatives: 2,449,029 rows of 41,000 representatives with 7 features
// 193 / 171, 64 395 / 351, 100 598 / 576, 256 1,083 / 1,021; 300,007 of 9,400 with 96 79 / 66.  A sixteenth as many representatives
// as rows, 2,449,029 with 33 376 / 369, 48 380 / 381; an eighth, with 48 411 / 426, 1,000,003 with 100 329 / 340, but 16 75 / 71;
// a quarter, 1,000,003 with 64 178 / 168, 128 357 / 352, 256 665 / 658, but 33 159 / 161, 48 165 / 168; half, 64 224 / 219, 256
// 760 / 762.)
bool keeps_bits_of_groups(int64_t rows, int64_t groups, int64_t F) {
    return rows >= (F <= 32 || F % 32 == 0 ? 4 : 16) * groups;
}

// rows[i] = act(reps[index[i]] + bias) with its gradients.  The ReLU mask of the gradient is kept as one bit
// per element of a row or of a representative, written by the kernel that produces the rows (the reference keeps the rows themselves:
// layer/CompressgnnReconstruct.py:16-22); without a ReLU nothing of the [N, F] output is needed again, and without a gradient
// no bits are (16 features, 10^6 rows: 13.6 us with those of the rows, 16.2 with those of the representatives, 12.5 without).
// Hooks on saved tensors are shown the bits of the rows: a row of words per row of the output, all of them written.
c10::optional<Tensor> reconstruct(Tensor reps, Tensor index, c10::optional<Tensor> bias, bool relu, Members members) {
    if (needs_function(reps, bias)) return c10::nullopt;
    Tensor rows, signs, ids;
    const bool with_bias = bias.has_value() && bias->defined();
    const bool recorded = at::GradMode::is_enabled() && (reps.requires_grad() || (with_bias && bias->requires_grad()));
    const bool hooks = !at::SavedTensorDefaultHooks::get_tls_state().stack.empty();
    const bool by_group = !hooks && reps.dim() == 2 && keeps_bits_of_groups(index.numel(), reps.size(0), reps.size(1));
    {
        at::AutoDispatchBelowADInplaceOrView plain;
        ids = index.contiguous();
        c10::optional<Tensor> b;
        if (with_bias) b = bias->contiguous();
        if (relu && recorded) std::tie(rows, signs) = by_group ? cluster_reconstruct_masks(reps.contiguous(), ids, b, members)
                                                   : cluster_reconstruct_signs(reps.contiguous(), ids, b, members);
        else rows = cluster_reconstruct(reps.contiguous(), ids, b, relu, members);
    }
    if (recorded) {
        auto node = with_bias ? node_over<ReconstructBackward>(reps, *bias) : node_over<ReconstructBackward>(reps);
        node->index = torch::autograd::SavedVariable(ids, false);
        if (relu) node->signs = torch::autograd::SavedVariable(signs, false);
        node->members = std::move(members);
        node->groups = reps.size(0);
        node->relu = relu;
        node->by_group = by_group;
        node->with_bias = with_bias;
        torch::autograd::set_history(rows, node);
    }
    return rows;
}

// (colptr, row, value) of a block held as int64 tensors on a GPU: the CSR of its transpose,
// in the order SparseTensor.csc() gives.  The one host read (a flag for columns out of
// range) comes after the last kernel.
std::tuple<Tensor, Tensor, c10::optional<Tensor>> csr_transpose(Tensor rowptr, Tensor col, c10::optional<Tensor> value,
                                                                int64_t cols) {
    TORCH_CHECK(rowptr.is_cuda() && col.is_cuda(), "csr_transpose: tensors must be on a GPU");
    TORCH_CHECK(rowptr.scalar_type() == torch::kInt64 && col.scalar_type() == torch::kInt64,
                "csr_transpose: rowptr and col must be int64");
    TORCH_CHECK(rowptr.dim() == 1 && col.dim() == 1 && rowptr.numel() >= 1 && cols >= 0, "csr_transpose: bad shapes");
    c10::hip::HIPGuardMasqueradingAsCUDA guard(rowptr.device());
    const int64_t rows = rowptr.numel() - 1, nnz = col.numel();
    Tensor rp = rowptr.contiguous(), ci = col.contiguous();
    Tensor val;
    int dtype = CGNN_F32;
    if (value.has_value() && value->defined()) {
        TORCH_CHECK(value->is_cuda() && value->dim() == 1 && value->numel() == nnz,
                    "csr_transpose: value must have one entry per non-zero");
        TORCH_CHECK(value->scalar_type() == torch::kFloat32 || value->scalar_type() == torch::kFloat64,
                    "csr_transpose: value must be float32 or float64");
        val = value->contiguous();
        dtype = dtype_code(val);
    }
    Tensor colptr = torch::empty({cols + 1}, rp.options());
    Tensor row = torch::empty({nnz}, rp.options());
    Tensor tval = val.defined() ? torch::empty_like(val) : Tensor();
    Tensor bad = torch::empty({1}, rp.options().dtype(torch::kInt32));
    const size_t bytes = cgnn_csr_transpose_workspace_bytes(nnz);
    Tensor ws = torch::empty({(int64_t)std::max<size_t>(bytes, 1)}, rp.options().dtype(torch::kUInt8));
    ok(cgnn_csr_transpose_device(rows, cols, nnz, rp.data_ptr<int64_t>(), nnz ? ci.data_ptr<int64_t>() : nullptr, dtype,
                                 val.defined() && nnz ? val.data_ptr() : nullptr, colptr.data_ptr<int64_t>(),
                                 nnz ? row.data_ptr<int64_t>() : nullptr, tval.defined() && nnz ? tval.data_ptr() : nullptr,
                                 bad.data_ptr<int32_t>(), ws.data_ptr(), bytes, current_stream(rp)),
       "csr_transpose");
    TORCH_CHECK(bad.item<int32_t>() == 0, "csr_transpose: column out of range [0, ", cols, ")");
    if (tval.defined()) return {colptr, row, tval};
    return {colptr, row, c10::nullopt};
}

// ------------------------------------------------ neighbour sampling (compressed graph) ----

// The host side of a sampling call: sizes the outputs of every layer (two scalar reads per
// layer: neighbours of the layer, vertices it adds) and strings the device entry points
// together.  neighbor_sample_sim_impl / neighbor_sample_ori_impl of the reference's module
// compressgnn_sample (src/sample/csrc/neighbor_sample.h:27-131, 134-211), on GPU tensors.
struct SampleGraph {
    cgnn_sample_graph view{};
    std::vector<Tensor> keep;  // contiguous int64 tensors behind the pointers
    torch::Device device = torch::kCPU;

    const int64_t *hold(const Tensor &t, const char *name) {
        TORCH_CHECK(t.defined() && t.is_cuda() && t.scalar_type() == torch::kInt64 && t.dim() == 1,
                    "neighbor_sample: ", name, " has to be a one-dimensional int64 GPU tensor");
        TORCH_CHECK(keep.empty() || t.device() == device, "neighbor_sample: ", name, " lives on another device");
        device = t.device();
        keep.push_back(t.contiguous());
        return keep.back().numel() ? keep.back().data_ptr<int64_t>() : nullptr;
    }
};

std::tuple<Tensor, Tensor, Tensor> run_sampler(SampleGraph &G, const Tensor &input_node,
                                               const std::vector<int64_t> &num_neighbors, int64_t seed, bool swap_roles) {
    const char *op = "neighbor_sample";
    const cgnn_sample_graph &g = G.view;
    TORCH_CHECK(input_node.is_cuda() && input_node.device() == G.device && input_node.scalar_type() == torch::kInt64 &&
                    input_node.dim() == 1,
                op, ": input_node has to be a one-dimensional int64 tensor beside the graph");
    for (int64_t fan : num_neighbors) TORCH_CHECK(fan >= 0, op, ": a fan-out of ", fan);
    c10::hip::HIPGuardMasqueradingAsCUDA guard(G.device);
    auto stream = current_stream(input_node);
    auto i64 = input_node.options();
    auto i32 = input_node.options().dtype(torch::kInt32);
    auto u8 = input_node.options().dtype(torch::kUInt8);
    const Tensor input = input_node.contiguous();
    const int64_t n_input = input.numel();
    auto raise_on = [&](int32_t code) {
        TORCH_CHECK_INDEX(code != CGNN_SAMPLE_OUT_OF_RANGE, "Neighbor index out of range");
        TORCH_CHECK(code != CGNN_SAMPLE_BAD_VERTEX, op, ": a vertex id outside [0, ", g.vertex_cnt, ")");
        TORCH_CHECK(code != CGNN_SAMPLE_TOO_MANY, op, ": a layer of more than 2^31 - 2 neighbours");
    };
    const int layers = (int)std::min<size_t>(num_neighbors.size(), INT_MAX);
    const size_t bounded = cgnn_sample_layers_workspace_bytes(g.vertex_cnt, n_input, layers, num_neighbors.data());
    Tensor slots;
    try {
        if (bounded > 0) slots = torch::empty({(int64_t)bounded}, u8);
    } catch (const c10::OutOfMemoryError &) {  // room for the longest lists there could be: the layers take what they are
    }
    if (slots.defined()) {
        const Tensor &ws = slots;
        const size_t bytes = bounded;
        Tensor summary = torch::empty({4}, torch::TensorOptions().dtype(torch::kInt32).pinned_memory(true));
        ok(cgnn_sample_layers(&g, n_input, input.data_ptr<int64_t>(), layers, num_neighbors.data(), (uint64_t)seed,
                              summary.data_ptr<int32_t>(), ws.data_ptr(), bytes, stream),
           op);
        const int32_t *sizes = summary.data_ptr<int32_t>();
        // a stream with little work ahead has them within this time
        await(sizes + 3, 0, kShortWait, stream, op);
        if (sizes[2] != -1) {  // -1: degrees that do not bound the lists; the layers then go one by one
            raise_on(sizes[2]);
            Tensor samples = torch::empty({sizes[0]}, i64), source = torch::empty({sizes[1]}, i64), neighbor = torch::empty({sizes[1]}, i64);
            ok(cgnn_sample_layers_write(&g, n_input, input.data_ptr<int64_t>(), layers, num_neighbors.data(), sizes[0], sizes[1],
                                        samples.data_ptr<int64_t>(), source.data_ptr<int64_t>(), neighbor.data_ptr<int64_t>(),
                                        ws.data_ptr(), bytes, stream),
               op);
            if (swap_roles) return {samples, neighbor, source};
            return {samples, source, neighbor};
        }
    }
    Tensor local_of = torch::empty({std::max<int64_t>(g.vertex_cnt, 1)}, i32), seen_at = torch::empty_like(local_of);
    Tensor status = torch::empty({1}, i32);
    ok(cgnn_sample_relabel_begin(g.vertex_cnt, n_input, n_input ? input.data_ptr<int64_t>() : nullptr,
                                 local_of.data_ptr<int32_t>(), seen_at.data_ptr<int32_t>(), status.data_ptr<int32_t>(),
                                 stream),
       op);
    Tensor samples = input.clone();
    std::vector<Tensor> sources, numbers;
    int64_t begin = 0, end = n_input;
    for (size_t layer = 0; layer < num_neighbors.size(); ++layer) {
        const int64_t n = end - begin, fanout = num_neighbors[layer];
        if (n == 0) break;
        Tensor frontier = samples.narrow(0, begin, n);
        Tensor counts = torch::empty({n}, i32), offsets = torch::empty({n + 1}, i32);
        ok(cgnn_sample_count(&g, n, frontier.data_ptr<int64_t>(), fanout, counts.data_ptr<int32_t>(),
                             status.data_ptr<int32_t>(), stream),
           op);
        const size_t sum_bytes = cgnn_exclusive_sum_workspace_bytes(n);
        Tensor sum_ws = torch::empty({(int64_t)std::max<size_t>(sum_bytes, 1)}, u8);
        ok(cgnn_exclusive_sum_i32(n, counts.data_ptr<int32_t>(), offsets.data_ptr<int32_t>(), status.data_ptr<int32_t>(),
                                  sum_ws.data_ptr(), sum_bytes, stream),
           op);
        // first scalar read of the layer: its size (and whether anything went wrong so far)
        Tensor head = torch::stack({offsets[n], status[0]}).cpu();
        raise_on(head.data_ptr<int32_t>()[1]);
        const int64_t total = head.data_ptr<int32_t>()[0];
        Tensor neighbors = torch::empty({total}, i64), source = torch::empty({total}, i64), picks = torch::empty({total}, i64);
        Tensor number = torch::empty({total}, i64), added = torch::empty({1}, i64);
        Tensor grown = torch::empty({end + total}, i64);
        grown.narrow(0, 0, end).copy_(samples);
        if (total > 0) {
            ok(cgnn_sample_fill(&g, n, frontier.data_ptr<int64_t>(), fanout, offsets.data_ptr<int32_t>(), begin,
                                (int64_t)layer, (uint64_t)seed, neighbors.data_ptr<int64_t>(), source.data_ptr<int64_t>(),
                                picks.data_ptr<int64_t>(), status.data_ptr<int32_t>(), stream),
               op);
        }
        const size_t bytes = cgnn_sample_relabel_workspace_bytes(total);
        Tensor ws = torch::empty({(int64_t)std::max<size_t>(bytes, 1)}, u8);
        ok(cgnn_sample_relabel(total, total ? neighbors.data_ptr<int64_t>() : nullptr, end, local_of.data_ptr<int32_t>(),
                               seen_at.data_ptr<int32_t>(), grown.data_ptr<int64_t>(), total ? number.data_ptr<int64_t>() : nullptr,
                               added.data_ptr<int64_t>(), ws.data_ptr(), bytes, stream),
           op);
        // second scalar read: how many vertices the layer added
        Tensor tail = torch::stack({added[0], status[0].to(torch::kInt64)}).cpu();
        raise_on((int32_t)tail.data_ptr<int64_t>()[1]);
        const int64_t fresh = tail.data_ptr<int64_t>()[0];
        samples = grown.narrow(0, 0, end + fresh);
        sources.push_back(source);
        numbers.push_back(number);
        begin = end;
        end += fresh;
    }
    Tensor empty = torch::empty({0}, i64);
    Tensor of_source = sources.empty() ? empty : torch::cat(sources), of_neighbor = numbers.empty() ? empty : torch::cat(numbers);
    // (samples, rows, cols): the compressed form reports (source, neighbour), the plain form the reverse
    if (swap_roles) return {samples.clone(), of_neighbor, of_source};
    return {samples.clone(), of_source, of_neighbor};
}

std::tuple<Tensor, Tensor, Tensor> neighbor_sample_cg_sim(Tensor v2v_vlist, Tensor v2v_elist, Tensor v2r_vlist,
                                                          Tensor v2r_elist, Tensor r2v_vlist, Tensor r2v_elist,
                                                          std::vector<Tensor> r2r_vlist, std::vector<Tensor> r2r_elist,
                                                          Tensor v_degree, Tensor r_degree, Tensor input_node,
                                                          std::vector<int64_t> num_neighbors, int64_t seed) {
    SampleGraph G;
    cgnn_sample_graph &g = G.view;
    g.v2v_ptr = G.hold(v2v_vlist, "v2v_vlist");
    g.v2v_idx = G.hold(v2v_elist, "v2v_elist");
    g.v2r_ptr = G.hold(v2r_vlist, "v2r_vlist");
    g.v2r_idx = G.hold(v2r_elist, "v2r_elist");
    g.r2v_ptr = G.hold(r2v_vlist, "r2v_vlist");
    g.r2v_idx = G.hold(r2v_elist, "r2v_elist");
    TORCH_CHECK(r2r_vlist.size() == r2r_elist.size() && r2r_vlist.size() <= CGNN_SAMPLE_MAX_LEVELS,
                "neighbor_sample: ", r2r_vlist.size(), " row-pointer and ", r2r_elist.size(), " column tensors of rule levels (at most ",
                CGNN_SAMPLE_MAX_LEVELS, " levels)");
    g.levels = (int32_t)r2r_vlist.size();
    g.vertex_cnt = v2v_vlist.numel() - 1;
    g.rule_cnt = r2v_vlist.numel() - 1;
    TORCH_CHECK(g.vertex_cnt >= 0 && g.rule_cnt >= 0 && v2r_vlist.numel() == g.vertex_cnt + 1,
                "neighbor_sample: row pointers have to hold vertex_cnt + 1 (v2v, v2r) and rule_cnt + 1 (r2v) entries");
    for (int k = 0; k < g.levels; ++k) {
        TORCH_CHECK(r2r_vlist[k].numel() == g.rule_cnt + 1, "neighbor_sample: level ", k, " has to hold rule_cnt + 1 row pointers");
        g.r2r_ptr[k] = G.hold(r2r_vlist[k], "r2r_vlist");
        g.r2r_idx[k] = G.hold(r2r_elist[k], "r2r_elist");
    }
    TORCH_CHECK(v_degree.numel() == g.vertex_cnt && r_degree.numel() == g.rule_cnt,
                "neighbor_sample: one expanded degree per vertex and per rule");
    g.v_degree = G.hold(v_degree, "v_degree");
    g.r_degree = G.hold(r_degree, "r_degree");
    return run_sampler(G, input_node, num_neighbors, seed, false);
}

std::tuple<Tensor, Tensor, Tensor> neighbor_sample_ori_impl(Tensor colptr, Tensor row, Tensor input_node,
                                                            std::vector<int64_t> num_neighbors, int64_t seed) {
    SampleGraph G;
    cgnn_sample_graph &g = G.view;
    g.v2v_ptr = G.hold(colptr, "colptr");
    g.v2v_idx = G.hold(row, "row");
    g.vertex_cnt = colptr.numel() - 1;
    TORCH_CHECK(g.vertex_cnt >= 0, "neighbor_sample: colptr has to hold vertex_cnt + 1 entries");
    return run_sampler(G, input_node, num_neighbors, seed, true);
}

// -------------------------------------------------------------- pair merger ----
// Arrays of the host cross to the device and back as int32 through pinned memory, a chunk at a time: all threads of the
// host check and convert (or copy) one while others are on their way, and the device takes up what has arrived.
// The 28 MB of int64 of a graph of 3.2 million edges took 0.4 ms to check and 0.7 ms to cross from pageable memory, and
// the 13 MB of result 0.95 ms; the link takes 0.25 ms either way.  kSlots chunks are in flight at most,
// whatever the size of the graph, and the pinned memory is the allocator's again after the call.
// Chunks take turns on two streams: behind a copy and its event the link is idle for 10 us if nothing else is there for it.
struct Link {
    static constexpr int64_t kChunk = 1 << 20, kSlots = 4;  // 4 MB: 76 us of the link, four times what they cost the host
    Tensor slots;
    hipStream_t streams[2];
    hipEvent_t sent[kSlots] = {}, ready = nullptr;

    // Copies come after the work that `compute` has been given so far.
    Link(int64_t most, c10::DeviceIndex device, hipStream_t compute) {
        for (auto &s : streams) s = c10::hip::getStreamFromPoolMasqueradingAsCUDA(false, device).stream();
        const int64_t n = std::max<int64_t>(1, std::min(kSlots * kChunk, most));
        slots = torch::empty({n}, torch::TensorOptions().dtype(torch::kInt32).pinned_memory(true));
        for (auto &e : sent) check(hipEventCreateWithFlags(&e, hipEventDisableTiming));
        check(hipEventCreateWithFlags(&ready, hipEventDisableTiming));
        check(hipEventRecord(ready, compute));
        for (auto &s : streams) check(hipStreamWaitEvent(s, ready, 0));
    }
    ~Link() {
        for (auto &s : streams) (void)hipStreamSynchronize(s);  // then nothing reads or writes the slots any more
        for (auto &e : sent)
            if (e != nullptr) (void)hipEventDestroy(e);
        if (ready != nullptr) (void)hipEventDestroy(ready);
    }
    Link(const Link &) = delete;
    static void check(hipError_t e) { TORCH_CHECK(e == hipSuccess, "compress_csr_batch: ", hipGetErrorString(e)); }
    int32_t *slot(int64_t k) { return slots.data_ptr<int32_t>() + k % kSlots * kChunk; }
    void copy(int64_t k, int32_t *to, const int32_t *from, int64_t n, hipMemcpyKind kind) {
        check(hipMemcpyAsync(to, from, n * sizeof(int32_t), kind, streams[k % 2]));
        check(hipEventRecord(sent[k % kSlots], streams[k % 2]));
    }
    void arrived(int64_t k) { check(hipEventSynchronize(sent[k % kSlots])); }
};

// The host's part of the way over a Link: work(chunk, at, n) for every block of kBlock entries of its chunks, by the
// calling thread and by helpers of torch's inter-op pool.  Blocks are handed out one by one, of the chunks opened so
// far, and nobody waits for a helper that has not begun: the calling thread does what is left.  (A parallel region
// of OpenMP waits at its end until all threads of its team have had a processor.  Behind a preparation step, whose own
// teams were still spinning, that cost 4 to 12 ms a region: calls took 2 to 97 ms there, and take 1.6 to 2.5 so; one
// after the other, with nothing else running, 1.27 ms with such regions and 1.33 so.)
class Crew {
    static constexpr int64_t kBlock = 1 << 14, kBlocks = Link::kChunk / kBlock;  // 10 us each
    static constexpr int kHelpers = 15;  // 3.2 million edges: 3 helpers 1.68 ms a call, 7 1.55, 11 1.49, 15 1.48
    struct Shared {
        std::function<void(int64_t, int64_t, int64_t)> work;
        std::vector<int64_t> entries;  // per chunk
        std::vector<std::atomic<int64_t>> left;
        std::atomic<int64_t> next{0}, open{0};
        std::atomic<int> inside{0};
        std::atomic<bool> stop{false};
        explicit Shared(size_t chunks) : left(chunks) {}

        bool one() {
            int64_t b = next.load();
            do
                if (b >= open.load() * kBlocks) return false;
            while (!next.compare_exchange_weak(b, b + 1));
            const int64_t chunk = b / kBlocks, at = b % kBlocks * kBlock, n = std::min(kBlock, entries[chunk] - at);
            if (n > 0) work(chunk, at, n);
            left[chunk].fetch_sub(1);
            return true;
        }
        // helper h calls helpers 2 h + 1 and 2 h + 2, so that the calling thread has one call to make (seven: 40 us)
        static void send(const std::shared_ptr<Shared> &s, int64_t h, int64_t helpers) {
            if (h < helpers)
                at::launch([s, h, helpers] {
                    send(s, 2 * h + 1, helpers);
                    send(s, 2 * h + 2, helpers);
                    s->help();
                });
        }
        void help() {
            ++inside;
            while (!stop.load() && next.load() < (int64_t)entries.size() * kBlocks)
                if (!one()) std::this_thread::yield();
            --inside;
        }
    };
    std::shared_ptr<Shared> shared;

public:
    Crew(std::vector<int64_t> entries, std::function<void(int64_t, int64_t, int64_t)> work)
        : shared(std::make_shared<Shared>(entries.size())) {
        int64_t blocks = 0;
        for (int64_t n : entries) blocks += (n + kBlock - 1) / kBlock;
        for (auto &l : shared->left) l = kBlocks;
        shared->entries = std::move(entries);
        shared->work = std::move(work);
        Shared::send(shared, 0, std::min<int64_t>({kHelpers, blocks / 2, at::get_num_threads() - 1, at::get_num_interop_threads()}));
    }
    ~Crew() {  // also where an error ends the call: no helper works on its arrays any more
        shared->stop = true;
        while (shared->inside.load() != 0) std::this_thread::yield();
    }
    Crew(const Crew &) = delete;
    void open(int64_t chunks) { shared->open = chunks; }
    void finish(int64_t chunk) {
        while (shared->left[chunk].load() != 0)
            if (!shared->one()) std::this_thread::yield();
    }
};

template <typename T>
bool narrow(const T *in, int64_t n, int32_t *out) {
    int64_t any = 0;
#pragma omp simd reduction(| : any)
    for (int64_t i = 0; i < n; ++i) {
        any |= (int64_t)in[i];
        out[i] = (int32_t)in[i];
    }
    return any >= 0 && any <= INT32_MAX;
}

// (row starts, columns, rules) of the compressed graph, as int32 tensors of the host.
std::tuple<Tensor, Tensor, int64_t> compress_csr_batch(const Tensor &vlist, const Tensor &elist, int64_t rounds,
                                                       int64_t min_pair_frequency) {
    const Tensor *in[2] = {&vlist, &elist};
    for (const Tensor *t : in)
        TORCH_CHECK(t->device().is_cpu() && t->dim() == 1 && t->is_contiguous() &&
                        (t->scalar_type() == torch::kInt64 || t->scalar_type() == torch::kInt32),
                    "compress_csr_batch: contiguous int64 or int32 arrays of the host");
    TORCH_CHECK_VALUE(rounds >= 1 && min_pair_frequency >= 3 && vlist.numel() > 0, "compress_csr_batch: bad arguments");
    const int64_t V = vlist.numel() - 1, E = elist.numel();
    const int passes = (int)std::min<int64_t>(rounds, INT_MAX), frequency = (int)std::min<int64_t>(min_pair_frequency, INT_MAX);
    auto done = [](int rc) {
        TORCH_CHECK_VALUE(rc != CGNN_EINVAL, cgnn_last_error());
        ok(rc, "compress_csr_batch");
    };
    struct Part {
        int array;
        int64_t at, n;
    };
    // the chunks of two arrays, one behind the other, and how many entries each has
    auto chunks_of = [](int64_t first, int64_t second, std::vector<int64_t> *entries) {
        std::vector<Part> parts;
        entries->clear();
        const int64_t n[2] = {first, second};
        for (int a = 0; a < 2; ++a)
            for (int64_t at = 0; at < n[a]; at += Link::kChunk) {
                parts.push_back({a, at, std::min(Link::kChunk, n[a] - at)});
                entries->push_back(parts.back().n);
            }
        return parts;
    };
    std::vector<int64_t> entries;
    const std::vector<Part> there = chunks_of(V + 1, E, &entries);
    // gone in the reverse order, also where an error ends the call: the helpers, the copies, what they copy
    Tensor dev[2], out_ptr, out_col, ws, result[2];
    std::unique_ptr<Link> up, down;
    std::atomic<bool> fits{true};
    // the helpers are on their way while the rest is made ready
    Crew sender(std::move(entries), [&](int64_t k, int64_t at, int64_t n) {
        const Tensor &from = *in[there[k].array];
        const int64_t first = there[k].at + at;
        if (!(from.scalar_type() == torch::kInt64 ? narrow(from.data_ptr<int64_t>() + first, n, up->slot(k) + at)
                                                  : narrow(from.data_ptr<int32_t>() + first, n, up->slot(k) + at)))
            fits = false;
    });
    const auto device = c10::Device(c10::kCUDA, c10::hip::current_device());
    const auto i32 = torch::TensorOptions().dtype(torch::kInt32).device(device);
    auto compute = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(device.index()).stream();
    auto stream = reinterpret_cast<cgnn_stream_t>(compute);
    const size_t bytes = cgnn_compress_batch_workspace_bytes(V, E);
    dev[0] = torch::empty({V + 1}, i32), dev[1] = torch::empty({std::max<int64_t>(E, 1)}, i32);
    out_ptr = torch::empty({V + E / 2 + 2}, i32), out_col = torch::empty({std::max<int64_t>(E, 1)}, i32);
    ws = torch::empty({(int64_t)std::max<size_t>(bytes, 1)}, i32.dtype(torch::kUInt8));
    up = std::make_unique<Link>(V + 1 + E + Link::kChunk, device.index(), compute);
    sender.open(std::min<int64_t>(there.size(), Link::kSlots));
    for (int64_t k = 0; k < (int64_t)there.size(); ++k) {
        if (k >= Link::kSlots) {
            up->arrived(k);  // the chunk whose slot this is
            sender.open(k + 1);
        }
        sender.finish(k);
        TORCH_CHECK_VALUE(fits, "CSR value exceeds int32 range");
        const auto [array, at, n] = there[k];
        int32_t *to = dev[array].data_ptr<int32_t>();
        up->copy(k, to + at, up->slot(k), n, hipMemcpyHostToDevice);
        Link::check(hipStreamWaitEvent(compute, up->sent[k % Link::kSlots], 0));
        if (array == 1) done(cgnn_compress_batch_feed(V, E, to, at, n, frequency, ws.data_ptr(), bytes, stream));
        else if (at + n == V + 1) done(cgnn_compress_batch_rows(V, E, to, frequency, ws.data_ptr(), bytes, stream));
    }
    Tensor pinned = torch::empty({9}, torch::TensorOptions().dtype(torch::kInt32).pinned_memory(true));
    int64_t summary[2] = {0, 0};
    done(cgnn_compress_batch_rounds(V, E, passes, frequency, out_ptr.data_ptr<int32_t>(), out_col.data_ptr<int32_t>(), summary,
                                    pinned.data_ptr<int32_t>(), ws.data_ptr(), bytes, stream));
    const std::vector<Part> back = chunks_of(V + summary[0] + 1, summary[1], &entries);
    const Tensor *from[2] = {&out_ptr, &out_col};
    Crew receiver(std::move(entries), [&](int64_t k, int64_t at, int64_t n) {
        std::memcpy(result[back[k].array].data_ptr<int32_t>() + back[k].at + at, down->slot(k) + at, n * sizeof(int32_t));
    });
    up.reset();
    const auto host = torch::TensorOptions().dtype(torch::kInt32);
    result[0] = torch::empty({V + summary[0] + 1}, host), result[1] = torch::empty({summary[1]}, host);
    down = std::make_unique<Link>(V + summary[0] + 1 + summary[1] + Link::kChunk, device.index(), compute);
    const int64_t n = (int64_t)back.size();
    for (int64_t k = 0; k < n + Link::kSlots; ++k) {
        if (const int64_t j = k - Link::kSlots; j >= 0 && j < n) {
            down->arrived(j);
            receiver.open(j + 1);
            receiver.finish(j);
        }
        if (k < n) down->copy(k, down->slot(k), from[back[k].array]->data_ptr<int32_t>() + back[k].at, back[k].n, hipMemcpyDeviceToHost);
    }
    return {result[0], result[1], summary[0]};
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    namespace py = pybind11;
    m.doc() = "CompressGNN runtime operators for MI355X (HIP kernels behind a C ABI)";
    // the reference's operator set (src/runtime/csrc/function.cpp:10-20)
    m.def("spmm_func", &spmm_func, "spmm function", py::arg("vlist"), py::arg("elist"), py::arg("value"),
          py::arg("mat"), py::arg("method"), py::arg("optional_out") = py::none());
    m.def("compress_csr_batch", &compress_csr_batch, py::arg("vlist"), py::arg("elist"), py::arg("rounds"),
          py::arg("min_pair_frequency"), py::call_guard<py::gil_scoped_release>());
    m.def("cluster_forward", &cluster_forward, "CompressGNN cluster forward");
    m.def("cluster_workspace", &cluster_workspace);
    m.def("cluster_assign", &cluster_assign);
    m.def("cluster_assign_members", &cluster_assign_members,
          "(ids, counts, active, [offsets, perm, sorted_id]) of one assignment refresh");
    m.def("cluster_mean", &cluster_mean, py::arg("input"), py::arg("index"), py::arg("count"),
          py::arg("members") = py::none());
    m.def("cluster_mean_backward", &cluster_mean_backward, py::arg("grad"), py::arg("index"), py::arg("count"),
          py::arg("members") = py::none());
    m.def("cluster_reconstruct", &cluster_reconstruct, py::arg("reps"), py::arg("index"), py::arg("bias"),
          py::arg("relu"), py::arg("members") = py::none());
    m.def("cluster_reconstruct_backward", &cluster_reconstruct_backward, py::arg("grad"), py::arg("index"),
          py::arg("output"), py::arg("groups"), py::arg("relu"), py::arg("members") = py::none());
    // the reference's sampler module (src/sample/csrc/function.cpp:7-9), here on GPU tensors; `seed` keys
    // the counter-based generator of the random positions
    m.def("neighbor_sample_cg_sim", &neighbor_sample_cg_sim, "Neighbor Sample with CompressGraph Format",
          py::arg("v2v_vlist"), py::arg("v2v_elist"), py::arg("v2r_vlist"), py::arg("v2r_elist"), py::arg("r2v_vlist"),
          py::arg("r2v_elist"), py::arg("r2r_vlist"), py::arg("r2r_elist"), py::arg("v_degree"), py::arg("r_degree"),
          py::arg("input_node"), py::arg("num_neighbors"), py::arg("seed") = 0);
    m.def("neighbor_sample_ori_impl", &neighbor_sample_ori_impl, "Neighbor Sample with Normal Graph Format",
          py::arg("colptr"), py::arg("row"), py::arg("input_node"), py::arg("num_neighbors"), py::arg("seed") = 0);
    // additions of this build
    m.def("cluster_members", &cluster_members, "member lists (offsets, perm, sorted_id) of the clusters");
    m.def("cluster_reconstruct_signs", &cluster_reconstruct_signs,
          "cluster_reconstruct with ReLU -> (rows, one sign bit per element)", py::arg("reps"), py::arg("index"),
          py::arg("bias"), py::arg("members") = py::none());
    m.def("cluster_reconstruct_backward_signs", &cluster_reconstruct_backward_signs,
          "cluster_reconstruct_backward with ReLU, masked by the sign bits", py::arg("grad"), py::arg("index"),
          py::arg("signs"), py::arg("groups"), py::arg("members") = py::none());
    m.def("cluster_reconstruct_masks", &cluster_reconstruct_masks,
          "cluster_reconstruct with ReLU -> (rows, one sign bit per element of a representative that has rows)", py::arg("reps"),
          py::arg("index"), py::arg("bias"), py::arg("members") = py::none());
    m.def("cluster_reconstruct_backward_masks", &cluster_reconstruct_backward_masks,
          "cluster_reconstruct_backward with ReLU, masked by the representatives' sign bits", py::arg("grad"), py::arg("index"),
          py::arg("masks"), py::arg("groups"), py::arg("members") = py::none());
    m.def("csr_transpose", &csr_transpose, "CSR -> CSC of an int64 block on the GPU, SparseTensor.csc() order",
          py::arg("rowptr"), py::arg("col"), py::arg("value"), py::arg("cols"));
    // the native steps of the layers: None under torch.jit.trace, for inputs with a tangent and under torch.func
    m.def("cluster_refresh", &cluster_refresh,
          "(representatives, ids, counts, active, [offsets, perm, sorted_id]) of an assignment refresh, with the gradient of "
          "the representatives", py::arg("x"), py::arg("planes"), py::arg("bits"));
    m.def("cluster_representatives", &cluster_representatives, "means over the clusters of an assignment, with their gradient",
          py::arg("x"), py::arg("index"), py::arg("counts"), py::arg("members"));
    m.def("reconstruct", &reconstruct, "act(reps[index] + bias) with its gradients", py::arg("reps"), py::arg("index"),
          py::arg("bias"), py::arg("relu"), py::arg("members") = py::none());
    m.def("column_sums", &column_sums, "sum over the rows of a matrix");
    m.def("propagate", &propagate, "plan.forward(x) with plan.backward as its gradient", py::arg("plan"), py::arg("x"),
          py::arg("once_differentiable") = false);
    m.def("version", []() { return std::string(cgnn_version()); });
    py::class_<DeviceCsr, std::shared_ptr<DeviceCsr>>(m, "DeviceCsr")
        .def(py::init([](Tensor rowptr, Tensor col, c10::optional<Tensor> value, int64_t rows, int64_t cols,
                         torch::Device device, int64_t seg_nnz, c10::optional<Tensor> rowmap, int64_t out_rows) {
                 return make_csr(rowptr, col, value, rows, cols, device, seg_nnz, rowmap, true, out_rows);
             }),
             py::arg("rowptr"), py::arg("col"), py::arg("value"), py::arg("rows"), py::arg("cols"),
             py::arg("device"), py::arg("seg_nnz") = 0, py::arg("rowmap") = py::none(), py::arg("out_rows") = -1)
        .def_readonly("rowmap", &DeviceCsr::rowmap)
        .def_readonly("out_rows", &DeviceCsr::out_rows)
        .def_readonly("rows", &DeviceCsr::rows)
        .def_readonly("cols", &DeviceCsr::cols)
        .def_readonly("nnz", &DeviceCsr::nnz)
        .def_readonly("max_row_nnz", &DeviceCsr::max_row_nnz)
        .def_property("seg_nnz", [](DeviceCsr &self) { return self.seg_nnz; },
                      [](DeviceCsr &self, int32_t seg) {
                          const std::shared_ptr<Scratch> scratch = self.scratch;
                          Hold hold(scratch->lock);
                          self.seg_nnz = seg;
                          self.run_start = Tensor();  // made again by the next product, like the workgroup runs
                          self.wg_runs.clear();
                          if (self.cut_rows.defined()) self.list_rows();  // the lists belong to a run length
                      })
        .def_readwrite("workgroup_runs", &DeviceCsr::workgroup_runs)
        .def_property_readonly("cut_rows", [](DeviceCsr &self) { return locked(self, &DeviceCsr::cut_rows); })
        .def_property_readonly("run_start", [](DeviceCsr &self) { return locked(self, &DeviceCsr::run_start); })
        .def_property_readonly("empty_rows", [](DeviceCsr &self) { return locked(self, &DeviceCsr::empty_rows); })
        .def_readonly("rowptr", &DeviceCsr::rowptr)
        .def_readonly("colidx", &DeviceCsr::colidx)
        .def_property_readonly("rowidx", [](DeviceCsr &self) { return locked(self, &DeviceCsr::rowidx); })
        .def_readonly("val", &DeviceCsr::val)
        .def("spmm",
             [](DeviceCsr &self, Tensor mat, c10::optional<Tensor> out, std::string method) {
                 return block_spmm(self, mat, out, kernel_of_method(method));
             },
             py::arg("mat"), py::arg("out") = py::none(), py::arg("method") = "auto");
    py::class_<PropagationPlan, std::shared_ptr<PropagationPlan>>(m, "PropagationPlan")
        .def(py::init([](int64_t V, int64_t R, std::shared_ptr<DeviceCsr> r2v, std::vector<std::shared_ptr<DeviceCsr>> r2r,
                         std::shared_ptr<DeviceCsr> v2r_t, std::vector<std::shared_ptr<DeviceCsr>> r2r_t) {
                 auto p = std::make_shared<PropagationPlan>();
                 TORCH_CHECK(r2v && v2r_t, "the rule stages r2v and v2r_t are required");
                 TORCH_CHECK(r2r.size() == r2r_t.size(), "levels and transposed levels differ in number");
                 TORCH_CHECK(r2v->rows == R && r2v->cols == V && v2r_t->rows == R && v2r_t->cols == V,
                             "the rule stages must be [rule_cnt, vertex_cnt]");
                 p->V = V; p->R = R;
                 p->r2v = r2v; p->r2r = r2r; p->v2r_t = v2r_t; p->r2r_t = r2r_t;
                 p->adopt(r2v); p->adopt(v2r_t);
                 for (auto &b : r2r) p->adopt(b);
                 for (auto &b : r2r_t) p->adopt(b);
                 return p;
             }),
             py::arg("vertex_cnt"), py::arg("rule_cnt"), py::arg("r2v"), py::arg("r2r"), py::arg("v2r_t"), py::arg("r2r_t"))
        .def("set_vertex_stages",
             [](PropagationPlan &p, std::shared_ptr<DeviceCsr> fwd, std::shared_ptr<DeviceCsr> bwd) {
                 TORCH_CHECK(fwd && bwd && fwd->rows == p.V && bwd->rows == p.V && fwd->cols == p.V + p.R &&
                                 bwd->cols == p.V + p.R,
                             "a vertex stage is [vertex_cnt, vertex_cnt + rule_cnt]");
                 std::array<MultipliedOut, 2> whole;
                 if (p.r2r.empty())  // no levels, or all of them in the rule stages
                     whole = surveyed({std::make_pair(fwd.get(), p.r2v.get()), std::make_pair(bwd.get(), p.v2r_t.get())}, p.V);
                 Hold hold(p.lock);
                 p.vertex_stage = fwd; p.vertex_stage_t = bwd;
                 p.whole = whole[0]; p.whole_t = whole[1];
                 p.composed.clear();
                 p.adopt(fwd); p.adopt(bwd);
             })
        .def("set_split_blocks",
             [](PropagationPlan &p, std::shared_ptr<DeviceCsr> v2v, std::shared_ptr<DeviceCsr> v2r,
                std::shared_ptr<DeviceCsr> v2v_t, std::shared_ptr<DeviceCsr> r2v_t) {
                 Hold hold(p.lock);
                 p.v2v = v2v; p.v2r = v2r; p.v2v_t = v2v_t; p.r2v_t = r2v_t;
                 p.adopt(v2v); p.adopt(v2r); p.adopt(v2v_t); p.adopt(r2v_t);
                 p.require_split_blocks();
             })
        .def_property("fuse_final", [](PropagationPlan &p) { return p.fuse_final; },
                      [](PropagationPlan &p, bool fuse) {
                          if (!fuse) p.require_split_blocks();
                          else TORCH_CHECK(p.vertex_stage && p.vertex_stage_t, "this plan has no fused vertex stages");
                          Hold hold(p.lock);
                          p.fuse_final = fuse;
                      })
        .def_readonly("vertex_stage", &PropagationPlan::vertex_stage)
        .def_readonly("vertex_stage_t", &PropagationPlan::vertex_stage_t)
        .def_property_readonly("scratch_bytes",
                               [](PropagationPlan &p) {
                                   Hold hold(p.scratch->lock);
                                   return p.scratch->buf.defined() ? p.scratch->buf.numel() : 0;
                               })
        .def_property("method",
                      [](PropagationPlan &p) { return p.kernel == CGNN_SPMM_ROW ? "row_schedule" : p.kernel == CGNN_SPMM_NNZ ? "nnz_schedule" : "auto"; },
                      [](PropagationPlan &p, std::string mth) {
                          Hold hold(p.lock);
                          p.kernel = kernel_of_method(mth);
                      })
        .def_property("timed_stages",
                      [](PropagationPlan &p) {
                          Hold hold(p.lock);
                          return p.timer.timed;
                      },
                      [](PropagationPlan &p, std::vector<std::string> names) {
                          Hold hold(p.lock);
                          p.timer.timed = names;
                      })
        .def_property("timed_every", [](PropagationPlan &p) { return p.timer.every; },
                      [](PropagationPlan &p, int64_t n) {
                          TORCH_CHECK(n >= 1, "timed_every must be at least 1");
                          Hold hold(p.lock);
                          p.timer.every = n;
                          p.timer.passes.clear();
                      })
        .def("take_stage_times",
             [](PropagationPlan &p) {
                 Hold hold(p.lock);
                 return p.timer.take();
             })
        .def_readonly("v2v", &PropagationPlan::v2v)
        .def_readonly("v2r", &PropagationPlan::v2r)
        .def_readonly("r2v", &PropagationPlan::r2v)
        .def_readonly("r2r", &PropagationPlan::r2r)
        .def_readonly("v2v_t", &PropagationPlan::v2v_t)
        .def_readonly("v2r_t", &PropagationPlan::v2r_t)
        .def_readonly("r2v_t", &PropagationPlan::r2v_t)
        .def_readonly("r2r_t", &PropagationPlan::r2r_t)
        .def("forward", &propagate_forward)
        .def("forward_gathered", &propagate_forward_gathered, py::arg("reps"), py::arg("index"),
             "out = A * reps[index] without the [vertex_cnt, F] matrix reps[index]")
        .def("backward", &propagate_backward);
}

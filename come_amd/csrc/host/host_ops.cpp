// The host side of the operators: argument checks, output allocation and the calls into libcome_hip.so, in native code.
//
// A merge or unmerge of one frame is 3 - 5 us of kernel, so what a call costs is the host path in front of the launch:
// through Python and ctypes a split took 11.4 us (about twenty interpreter-level tensor calls and a 20-argument foreign
// call); here it is one call that allocates through the caching allocator directly and launches.  The C ABI of
// libcome_hip.so stays the product's boundary: this module looks its functions up in the library the Python binding has
// loaded (bind) and knows nothing of its kernels.
//
// The packed row count of a merge decides the shape of its outputs, so it has to reach the host.  The plan kernels store
// it into pinned host memory (a Mailbox slot) while they run; the host polls that word.  A context whose mask was selected by
// rank from fp32 confidences knows how many windows merge unless window means tie at the threshold: the merge is then
// launched at once, with outputs of the expected size, and the posted count confirms it afterwards.
//
// Every merge finds its packed positions in the mask it is given.  A plan kept from the selection would spare that, but nothing
// tells the host that it still fits: collectives, other libraries' kernels and replayed graphs write a mask without a trace.
// Where the count is known but for ties the merge kernels need no plan at all (merge_direct).
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/PyInterpreter.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/csrc/utils/pybind.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/TensorSubclassLikeUtils.h>
#include <ATen/autocast_mode.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <dlfcn.h>
#include <hip/hip_runtime_api.h>

#include <chrono>
#include <cmath>
#include <mutex>
#include <optional>
#include <string>
#include <tuple>
#include <vector>

#include "../../../include/come_hip.h"

namespace py = pybind11;
using at::Tensor;

namespace {

// ---- libcome_hip.so -------------------------------------------------------------------------------------------
#define COME_FUNCTIONS(F)                                                                                         \
    F(come_last_error) F(come_merge_plan_post) F(come_token_merge_wide) F(come_token_merge_is_direct) F(come_token_merge_direct) F(come_token_split) F(come_token_split_pair) \
    F(come_select_plan_post) F(come_select_windows) F(come_attn_work_bytes) \
    F(come_attn_varlen_fwd_ws) F(come_qk_norm_rope) F(come_jagged_add_suffix)            \
    F(come_jagged_split_suffix_post) F(come_residual_norm) F(come_linear) F(come_linear_is_faster) \
    F(come_linear_splits) F(come_linear_split) F(come_residual_norm_split)
struct Abi {
#define F(name) decltype(&::name) name = nullptr;
    COME_FUNCTIONS(F)
#undef F
} abi;

void bind(uintptr_t library) {
    void *lib = reinterpret_cast<void *>(library);
#define F(name)                                                                          \
    abi.name = reinterpret_cast<decltype(abi.name)>(dlsym(lib, #name));                  \
    if (abi.name == nullptr) throw std::runtime_error("libcome_hip.so does not export " #name);
    COME_FUNCTIONS(F)
#undef F
}

void check(int status) {
    if (status == COME_OK) return;
    const char *msg = abi.come_last_error();
    throw std::runtime_error(msg && *msg ? std::string(msg) : "libcome_hip call failed with status " + std::to_string(status));
}
void require(bool cond, const char *msg) {
    if (!cond) throw std::runtime_error(msg);
}

int dtype_code(at::ScalarType t) {
    switch (t) {
        case at::kFloat: return COME_F32;
        case at::kHalf: return COME_F16;
        case at::kBFloat16: return COME_BF16;
        default:
            throw std::runtime_error(std::string("come_amd: unsupported dtype ") + c10::toString(t) +
                                     " (float32, float16, bfloat16 only)");
    }
}

// straight to the caching allocator of the tensors' device (which is current)
Tensor empty(at::IntArrayRef sizes, at::ScalarType dtype, const at::Device &dev) {
    return at::detail::empty_cuda(sizes, dtype, dev, std::nullopt);
}
hipStream_t stream_of(const at::Device &dev) {
    return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(dev.index()).stream();
}
template <typename T> T *data(const Tensor &t) { return static_cast<T *>(t.data_ptr()); }

// ---- mailbox: words of pinned host memory that kernels post one value into ----------------------------------------
// One page for the process, handed out a word at a time; a word goes back when what was posted to it has been seen, so no
// kernel still running can write into a word that somebody else waits for.  A call that ends without reading leaves its word
// on the waiting list until the post has arrived.  Without a free word (512 calls at a time) the count is read back instead.
class Mailbox {
public:
    static constexpr int kWords = 512;
    struct Slot {
        int index = -1;
        uint32_t tag = 0;
    };

    Slot take() {
        std::lock_guard<std::mutex> guard(lock_);
        if (words_ == nullptr && !failed_) {
            void *p = nullptr;
            if (hipHostMalloc(&p, kWords * sizeof(uint64_t), hipHostMallocMapped | hipHostMallocPortable | hipHostMallocCoherent) == hipSuccess) {
                words_ = static_cast<uint64_t *>(p);
                for (int i = 0; i < kWords; ++i) {
                    words_[i] = 0;
                    free_.push_back(i);
                }
            } else {
                (void)hipGetLastError();
                failed_ = true;
            }
        }
        if (free_.empty())
            for (size_t i = 0; i < unread_.size();) {
                if (arrived(unread_[i])) {
                    free_.push_back(unread_[i].index);
                    unread_[i] = unread_.back();
                    unread_.pop_back();
                } else {
                    ++i;
                }
            }
        Slot s;
        if (free_.empty()) return s;
        s.index = free_.back();
        free_.pop_back();
        if (++next_tag_ == 0) next_tag_ = 1;            // the words start as tag 0
        s.tag = next_tag_;
        return s;
    }
    void give_back(const Slot &s) {
        if (s.index < 0) return;
        std::lock_guard<std::mutex> guard(lock_);
        if (arrived(s)) free_.push_back(s.index);
        else unread_.push_back(s);
    }
    void give_back_unused(const Slot &s) {              // nothing was launched that could post to it
        if (s.index < 0) return;
        std::lock_guard<std::mutex> guard(lock_);
        free_.push_back(s.index);
    }
    uint64_t *word(const Slot &s) const { return s.index < 0 ? nullptr : words_ + s.index; }
    bool read(const Slot &s, uint32_t &value) const {
        const uint64_t v = __atomic_load_n(words_ + s.index, __ATOMIC_ACQUIRE);
        value = static_cast<uint32_t>(v);
        return static_cast<uint32_t>(v >> 32) == s.tag;
    }
    // Waits for the post of a launch on `stream`.  False: the stream has run dry (or failed) without it.
    bool wait(const Slot &s, hipStream_t stream, uint32_t &value) const {
        if (s.index < 0) return false;
        for (int i = 0; i < 64; ++i)
            if (read(s, value)) return true;
        py::gil_scoped_release release;
        auto next_look = std::chrono::steady_clock::now() + std::chrono::microseconds(200);
        for (;;) {
            for (int i = 0; i < 64; ++i) {
                if (read(s, value)) return true;
                __builtin_ia32_pause();
            }
            if (std::chrono::steady_clock::now() < next_look) continue;
            if (hipStreamQuery(stream) != hipErrorNotReady) {
                (void)hipGetLastError();
                return read(s, value);
            }
            next_look = std::chrono::steady_clock::now() + std::chrono::microseconds(200);
        }
    }

private:
    bool arrived(const Slot &s) const {
        uint32_t v;
        return read(s, v);
    }
    std::mutex lock_;
    uint64_t *words_ = nullptr;
    bool failed_ = false;
    uint32_t next_tag_ = 0;
    std::vector<int> free_;
    std::vector<Slot> unread_;
};
Mailbox &mailbox() {
    static Mailbox *m = new Mailbox;                    // never destroyed: kernels may outlive static destruction
    return *m;
}

bool recording(hipStream_t stream) {
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &status) == hipSuccess) return status != hipStreamCaptureStatusNone;
    (void)hipGetLastError();                            // (the default stream beside another one's capture)
    return true;
}

// What one launch posts.  Its word goes back when the value has been seen or, where nothing was launched, at once.  A launch
// that is being recorded gets none: every replay would post the same tag, long after the word belongs to somebody else.
class Post {
public:
    explicit Post(hipStream_t stream) : stream_(stream) {
        if (!recording(stream)) slot_ = mailbox().take();
    }
    Post(const Post &) = delete;
    Post &operator=(const Post &) = delete;
    ~Post() {
        if (launched_) mailbox().give_back(slot_);
        else mailbox().give_back_unused(slot_);
    }
    uint64_t *word() const { return mailbox().word(slot_); }
    uint32_t tag() const { return slot_.tag; }
    void launched() { launched_ = true; }
    bool wait(uint32_t &value) const { return launched_ && mailbox().wait(slot_, stream_, value); }

private:
    Mailbox::Slot slot_;
    hipStream_t stream_;
    bool launched_ = false;
};

// ---- merge plan -------------------------------------------------------------------------------------------------
// From a merge mask to packed positions.
class MergePlan {
public:
    const int64_t rows, groups, start, group_size, tail;
    Tensor offsets;                                     // int32 [rows + 1]

    MergePlan(const at::Device &dev, int64_t rows_, int64_t groups_, int64_t start_, int64_t group_size_, int64_t tail_)
        : rows(rows_), groups(groups_), start(start_), group_size(group_size_), tail(tail_), stream_(stream_of(dev)), count_(stream_) {
        // (the prefix starts at a multiple of 16 bytes)
        const int64_t n_off = (rows + 1 + 3) / 4 * 4;
        const Tensor both = empty({n_off + std::max<int64_t>(rows * groups, 1)}, at::kInt, dev);
        offsets = both.narrow(0, 0, rows + 1);
        prefix_ = data<int32_t>(both) + n_off;
    }
    void make(const Tensor &mask) {
        check(abi.come_merge_plan_post(mask.numel() > 0 ? data<uint8_t>(mask) : nullptr, rows, groups, start, group_size, tail,
                                       data<int32_t>(offsets), prefix_, count_.word(), count_.tag(), stream_));
        count_.launched();
    }
    int32_t *prefix() const { return prefix_; }
    hipStream_t stream() const { return stream_; }
    Post &count() { return count_; }
    // Packed rows: posted by the plan's launch, read back from the offsets where there was no word for it.
    int64_t packed_rows() {
        uint32_t v = 0;
        if (rows == 0) return 0;
        return count_.wait(v) ? v : offsets.select(0, rows).item<int32_t>();
    }

private:
    hipStream_t stream_;
    Post count_;
    int32_t *prefix_ = nullptr;
};

// Windows that merge where `batch` elements of n windows each are selected by rank from distinct fp32 means, -1: not known.
// With q = quantile(means, threshold), floor(rank) + 1 of distinct means lie below it, floor(rank) where the rank is a whole
// number (q is then one of the means).  bf16 means tie all the time: nothing is expected of them.
int64_t expected_windows(int mode, at::ScalarType dtype, int64_t batch, int64_t n, double threshold) {
    if (mode != 0 || dtype != at::kFloat) return -1;
    const float rank = static_cast<float>(threshold) * static_cast<float>(n - 1);
    const float low = std::floor(rank);
    return batch * (static_cast<int64_t>(low) + (rank > low ? 1 : 0));
}

void check_confidence(const Tensor &confidence) {
    require(confidence.is_cuda(), "conf must be on CUDA");
    require(confidence.scalar_type() == at::kBFloat16 || confidence.scalar_type() == at::kFloat, "conf must be bfloat16 or float32");
}

// confidence -> (mask, windows expected to merge or -1).  The grid holds at least one full window.
std::tuple<Tensor, int64_t> select_mask(const Tensor &confidence, int64_t batch, int64_t rows, int64_t H, int64_t W, int64_t gh,
                                   int64_t gw, double threshold, int mode) {
    check_confidence(confidence);
    const Tensor conf = confidence.contiguous();
    const at::Device dev = conf.device();
    c10::DeviceGuard guard(dev);
    const int64_t M = (H / gh) * (W / gw);
    Tensor mask = empty({rows, M}, at::kBool, dev);
    const Tensor means = empty({rows, M}, at::kFloat, dev);
    check(abi.come_select_windows(conf.data_ptr(), dtype_code(conf.scalar_type()), batch, rows / batch, H, W, gh, gw, mode,
                                  static_cast<float>(threshold), data<float>(means), data<uint8_t>(mask), nullptr, 0, stream_of(dev)));
    return {mask, expected_windows(mode, conf.scalar_type(), batch, rows / batch * M, threshold)};
}

struct Merged {
    Tensor out, offsets32, offsets64, index_map, counts;
};

// tokens [rows, n_tok, C] (or [B, S, n_tok, C]), contiguous; plan: of `mask`, launched in this call; expected: windows that
// probably merge, or -1; lead: shape of the packed tensor, [1, P, C] or [P, C]
Merged merge(const Tensor &tokens, int64_t rows, int64_t n_tok, int64_t C, int64_t start, int64_t gh, int64_t gw, int64_t H,
             int64_t W, const Tensor &mask, MergePlan &plan, int64_t expected, at::ScalarType index_dtype,
             at::ScalarType count_dtype, bool wide, bool lead) {
    const at::Device dev = tokens.device();
    const int code = dtype_code(tokens.scalar_type());
    Merged m;
    m.offsets32 = plan.offsets;
    m.index_map = empty({rows * n_tok}, index_dtype, dev);
    if (wide) m.offsets64 = empty({rows + 1}, at::kLong, dev);
    auto launch = [&](int64_t P) {
        m.out = lead ? empty({1, P, C}, tokens.scalar_type(), dev) : empty({P, C}, tokens.scalar_type(), dev);
        m.counts = empty({P}, count_dtype, dev);
        void *index = m.index_map.data_ptr(), *counts = m.counts.data_ptr();
        check(abi.come_token_merge_wide(
            tokens.data_ptr(), code, rows, n_tok, C, start, gh, gw, H, W, mask.numel() > 0 ? data<uint8_t>(mask) : nullptr,
            data<int32_t>(plan.offsets), plan.prefix(), m.out.data_ptr(), P,
            index_dtype == at::kLong ? static_cast<int64_t *>(index) : nullptr,
            index_dtype == at::kInt ? static_cast<int32_t *>(index) : nullptr,
            count_dtype == at::kFloat ? static_cast<float *>(counts) : nullptr,
            count_dtype == at::kInt ? static_cast<int32_t *>(counts) : nullptr, wide ? data<int64_t>(m.offsets64) : nullptr,
            plan.stream()));
    };
    const int64_t guess = expected >= 0 && expected <= plan.rows * plan.groups ? rows * n_tok - expected * (plan.group_size - 1) : 0;
    if (guess > 0) launch(guess);                        // (rows beyond the outputs are not written)
    const int64_t P = plan.packed_rows();
    if (P != guess || guess == 0) launch(P);             // means tied at the threshold, or the mask has been written to
    if (wide && (rows == 0 || n_tok == 0)) m.offsets64 = plan.offsets.to(at::kLong);      // nothing was launched
    return m;
}

// A merge whose packed row count is known but for ties, straight from the mask: one launch, which posts the count.  Nothing:
// the kernels do not take it, or there is no word to post to (while recording); the merge is planned first then.
std::optional<Merged> merge_direct(const Tensor &tokens, int64_t rows, int64_t n_tok, int64_t C, int64_t start, int64_t gh, int64_t gw,
                                   int64_t H, int64_t W, const Tensor &mask, int64_t expected) {
    const at::Device dev = tokens.device();
    const int code = dtype_code(tokens.scalar_type());
    const int64_t guess = rows * n_tok - expected * (gh * gw - 1);
    if (expected < 0 || expected > mask.numel() || mask.numel() == 0 || guess <= 0 ||
        !abi.come_token_merge_is_direct(tokens.data_ptr(), code, rows, n_tok, C, gh, gw, H, W, data<uint8_t>(mask)))
        return std::nullopt;
    const hipStream_t stream = stream_of(dev);
    Post count(stream);
    if (count.word() == nullptr) return std::nullopt;
    Merged m;
    m.index_map = empty({rows * n_tok}, at::kLong, dev);
    m.offsets64 = empty({rows + 1}, at::kLong, dev);
    auto launch = [&](int64_t P, uint64_t *word) {
        m.out = empty({1, P, C}, tokens.scalar_type(), dev);
        m.counts = empty({P}, at::kFloat, dev);
        check(abi.come_token_merge_direct(tokens.data_ptr(), code, rows, n_tok, C, start, gh, gw, H, W, data<uint8_t>(mask), m.out.data_ptr(),
                                          P, data<int64_t>(m.index_map), nullptr, data<float>(m.counts), nullptr,
                                          data<int64_t>(m.offsets64), word, count.tag(), stream));
    };
    launch(guess, count.word());
    count.launched();
    uint32_t posted = 0;
    const int64_t P = count.wait(posted) ? posted : m.offsets64.select(0, rows).item<int64_t>();
    if (P != guess) launch(P, nullptr);                  // means tied at the threshold, or the mask has been written to
    return m;
}

// ---- token merger entry points.  None: the arguments are not what the operator takes; the caller's checks say why. ----
py::object merge_2d(const Tensor &tokens, int64_t start, int64_t gh, int64_t gw, int64_t H, int64_t W, const Tensor &mask,
                    bool allow_remainder, int64_t expected) {
    const int64_t d = tokens.dim();
    if (d != 3 && d != 4) return py::none();
    const int64_t rows = d == 4 ? tokens.size(0) * tokens.size(1) : tokens.size(0), n_tok = tokens.size(d - 2), C = tokens.size(d - 1);
    if (!tokens.is_cuda() || !mask.is_cuda() || mask.scalar_type() != at::kBool || mask.dim() != 2 || start < 0 || gh <= 0 || gw <= 0 ||
        H < 0 || W < 0 || (!allow_remainder && (H % gh != 0 || W % gw != 0)) || mask.size(0) != rows || n_tok != start + H * W ||
        mask.size(1) != (H / gh) * (W / gw) || mask.device() != tokens.device())
        return py::none();
    c10::DeviceGuard guard(tokens.device());
    const Tensor tok = tokens.contiguous(), merged = mask.contiguous();
    if (const auto m = merge_direct(tok, rows, n_tok, C, start, gh, gw, H, W, merged, expected))
        return py::make_tuple(m->out, m->counts, m->offsets64, m->index_map);
    MergePlan plan(tokens.device(), rows, mask.size(1), start, gh * gw, H * W - mask.size(1) * gh * gw);
    plan.make(merged);
    const Merged m = merge(tok, rows, n_tok, C, start, gh, gw, H, W, merged, plan, expected, at::kLong, at::kFloat, true, true);
    return py::make_tuple(m.out, m.counts, m.offsets64, m.index_map);
}

py::object merge_1d(const Tensor &tokens, int64_t start, int64_t G, const Tensor &mask, bool wide) {
    if (tokens.dim() != 3 || mask.dim() != 2 || !tokens.is_cuda() || !mask.is_cuda() || mask.scalar_type() != at::kBool || start < 0 ||
        G <= 0 || mask.size(0) != tokens.size(0) || tokens.size(1) != start + mask.size(1) * G || mask.device() != tokens.device())
        return py::none();
    c10::DeviceGuard guard(tokens.device());
    const int64_t M = mask.size(1);
    const Tensor tok = tokens.contiguous(), merged = mask.contiguous();
    MergePlan plan(tokens.device(), tokens.size(0), M, start, G, 0);
    plan.make(merged);
    const Merged m = merge(tok, tokens.size(0), tokens.size(1), tokens.size(2), start, 1, G, M > 0 ? 1 : 0, M * G, merged, plan, -1,
                           at::kLong, at::kFloat, wide, wide);
    return py::make_tuple(m.out, wide ? m.offsets64 : m.offsets32, m.index_map, m.counts);
}

// the operator with the caller's index and count types: (out [P, C], offsets int32, index_map, counts)
py::tuple merge_2d_flat(const Tensor &tokens, int64_t start, int64_t gh, int64_t gw, int64_t H, int64_t W, const Tensor &mask,
                        bool index_64, bool count_float) {
    c10::DeviceGuard guard(tokens.device());
    const Tensor tok = tokens.contiguous(), merged = mask.contiguous();
    const int64_t M = (H / gh) * (W / gw);
    MergePlan plan(tokens.device(), mask.size(0), M, start, gh * gw, H * W - M * gh * gw);
    plan.make(merged);
    const Merged m = merge(tok, tokens.size(0), tokens.size(1), tokens.size(2), start, gh, gw, H, W, merged, plan, -1,
                           index_64 ? at::kLong : at::kInt, count_float ? at::kFloat : at::kInt, false, false);
    return py::make_tuple(m.out, m.offsets32, m.index_map, m.counts);
}

// confidence -> mask and plan in one launch, and the merge behind it: (out [P, C], index_map, counts, offsets int32, mask).  The
// grid holds at least one full window.
py::tuple select_merge_2d(const Tensor &tokens, const Tensor &confidence, int64_t batch, int64_t start, int64_t gh, int64_t gw,
                          int64_t H, int64_t W, double threshold, int mode, bool index_64, bool count_float) {
    check_confidence(confidence);
    const Tensor tok = tokens.contiguous(), conf = confidence.contiguous();
    const at::Device dev = tokens.device();
    c10::DeviceGuard guard(dev);
    const int64_t rows = tokens.size(0), M = (H / gh) * (W / gw), n = rows / batch * M;
    const Tensor mask = empty({rows, M}, at::kBool, dev);
    MergePlan plan(dev, rows, M, start, gh * gw, H * W - M * gh * gw);
    Tensor means;
    if (n > 16384) means = empty({batch * n}, at::kFloat, dev);          // fewer keys stay in the workgroup's LDS
    check(abi.come_select_plan_post(
        conf.data_ptr(), dtype_code(conf.scalar_type()), batch, rows / batch, H, W, gh, gw, mode, static_cast<float>(threshold), start,
        means.defined() ? data<float>(means) : nullptr, data<uint8_t>(mask), data<int32_t>(plan.offsets), plan.prefix(), nullptr, 0,
        plan.count().word(), plan.count().tag(), plan.stream()));
    plan.count().launched();
    const Merged m = merge(tok, rows, tokens.size(1), tokens.size(2), start, gh, gw, H, W, mask, plan,
                           expected_windows(mode, conf.scalar_type(), batch, n, threshold), index_64 ? at::kLong : at::kInt,
                           count_float ? at::kFloat : at::kInt, false, false);
    return py::make_tuple(m.out, m.index_map, m.counts, m.offsets32, mask);
}

// ---- unmerge ----------------------------------------------------------------------------------------------------
// merged [P, C] or [1, P, C]; `shape`: of the result, whose last dimension is C (or 2 C with a second source)
Tensor split(const Tensor &a, const std::optional<Tensor> &b, const Tensor &rev, int64_t C, std::vector<int64_t> shape) {
    const bool pair = b.has_value();
    require(a.is_cuda() && (!pair || b->is_cuda()), pair ? "merged_a and merged_b must be on CUDA" : "merged_flat must be on CUDA");
    require(rev.is_cuda(), "rev_id must be on CUDA");
    const bool flat = a.dim() == 2 || (a.dim() == 3 && a.size(0) == 1);
    if (pair) {
        require(flat && a.size(-1) == C, "merged_a must be [P, C]");
        require(b->sizes() == a.sizes() && b->scalar_type() == a.scalar_type() && b->device() == a.device(),
                "merged_b must match merged_a in shape, dtype and device");
    } else {
        require(flat, "merged_flat must be [P, C]");
        require(a.size(-1) == C, "C mismatch");
    }
    const auto index = rev.scalar_type();
    require(index == at::kLong || index == at::kInt, "rev_id must be int64 or int32");
    const Tensor a_c = a.contiguous(), rev_c = rev.contiguous();
    const Tensor b_c = pair ? b->contiguous() : Tensor();
    const int64_t total = rev_c.numel(), P = a_c.size(-2);
    const at::Device dev = a_c.device();
    c10::DeviceGuard guard(dev);
    if (shape.empty()) shape = {total, pair ? 2 * C : C};
    int64_t elements = 1;
    for (int64_t s : shape) elements *= s;
    require(elements == total * (pair ? 2 * C : C), "rev_id does not hold one index per row of the result");
    Tensor out = empty(shape, a_c.scalar_type(), dev);
    const int64_t *r64 = index == at::kLong ? data<int64_t>(rev_c) : nullptr;
    const int32_t *r32 = index == at::kInt ? data<int32_t>(rev_c) : nullptr;
    const int code = dtype_code(a_c.scalar_type());
    if (pair)
        check(abi.come_token_split_pair(a_c.data_ptr(), b_c.data_ptr(), code, P, C, r64, r32, total, out.data_ptr(), stream_of(dev)));
    else
        check(abi.come_token_split(a_c.data_ptr(), code, P, C, r64, r32, total, out.data_ptr(), stream_of(dev)));
    return out;
}

// ---- attention --------------------------------------------------------------------------------------------------
// Packed self-attention with the plain options, for what the kernels take as it is (head widths 32, 64, 128; aligned
// views).  None: something is out of the ordinary, and the general path with its messages has to look at it.
std::optional<Tensor> attention(const Tensor &qkv, const Tensor &cu, int64_t max_seqlen, const std::optional<Tensor> &bias,
                                double scale, int flags) {
    const auto dtype = qkv.scalar_type();
    if (!qkv.is_cuda() || (dtype != at::kBFloat16 && dtype != at::kHalf) || qkv.dim() != 4 || qkv.size(1) != 3) return std::nullopt;
    const int64_t total = qkv.size(0), H = qkv.size(2), D = qkv.size(3);
    const at::Device dev = qkv.device();
    if ((D != 32 && D != 64 && D != 128) || H < 1 || total < 1 || max_seqlen < 2 || qkv.stride(3) != 1 || qkv.stride(0) % 8 != 0 ||
        qkv.stride(1) % 8 != 0 || qkv.stride(2) % 8 != 0 || reinterpret_cast<uintptr_t>(qkv.data_ptr()) % 16 != 0)
        return std::nullopt;
    if (!cu.is_cuda() || cu.scalar_type() != at::kInt || cu.dim() != 1 || !cu.is_contiguous() || cu.numel() < 2 || cu.device() != dev)
        return std::nullopt;
    if (bias && (bias->scalar_type() != dtype || !bias->is_cuda() || !bias->is_contiguous() || bias->dim() != 1 ||
                 bias->size(0) != total || bias->device() != dev))
        return std::nullopt;
    c10::DeviceGuard guard(dev);
    Tensor out = empty({total, H, D}, dtype, dev);
    const int64_t n_seq = cu.numel() - 1;
    const int64_t work_bytes = D == 64 ? abi.come_attn_work_bytes(n_seq, total, H, max_seqlen) : 0;
    Tensor work;
    if (work_bytes > 0) work = empty({work_bytes}, at::kByte, dev);
    const int64_t rs = qkv.stride(0), hs = qkv.stride(2), part = qkv.stride(1) * 2;          // (bytes between q, k and v)
    const char *q = data<char>(qkv);
    check(abi.come_attn_varlen_fwd_ws(q, q + part, q + 2 * part, dtype_code(dtype), rs, hs, rs, hs, rs, hs, data<int32_t>(cu), n_seq,
                                      total, H, D, bias ? bias->data_ptr() : nullptr, max_seqlen, static_cast<float>(scale),
                                      out.data_ptr(), H * D, D, nullptr, work_bytes > 0 ? work.data_ptr() : nullptr, work_bytes,
                                      flags, stream_of(dev)));
    return out;
}

// ---- q / k prologue ----------------------------------------------------------------------------------------------
// In place on the packed projection.  The parameters are taken as they are where they already have the run dtype.
// False: not a plain call (the general path converts, or says what is wrong).
bool qk_norm_rope(const Tensor &qkv, bool k_only, bool apply, double eps, const std::optional<Tensor> &qw, const std::optional<Tensor> &qb,
                  const std::optional<Tensor> &kw, const std::optional<Tensor> &kb, const std::optional<Tensor> &pos,
                  const std::optional<Tensor> &cos_table, const std::optional<Tensor> &sin_table, int64_t n_pos) {
    const auto dtype = qkv.scalar_type();
    const at::Device dev = qkv.device();
    const int64_t P = qkv.size(0), H = qkv.size(2), D = qkv.size(3);
    for (const auto *p : {&qw, &qb, &kw, &kb})
        if (p->has_value() && ((*p)->scalar_type() != dtype || (*p)->device() != dev || !(*p)->is_contiguous() || (*p)->numel() != D))
            return false;
    if (pos && (pos->scalar_type() != at::kLong || pos->device() != dev || !pos->is_contiguous() || pos->numel() != 2 * P)) return false;
    c10::DeviceGuard guard(dev);
    auto ptr = [](const std::optional<Tensor> &t) { return t ? t->data_ptr() : nullptr; };
    char *q = data<char>(qkv);
    check(abi.come_qk_norm_rope(k_only ? nullptr : q, q + 2 * qkv.stride(1), dtype_code(dtype), qkv.stride(0), qkv.stride(2), qkv.stride(0), qkv.stride(2), P,
                                H, D, apply ? 1 : 0, ptr(qw), ptr(qb), ptr(kw), ptr(kb), static_cast<float>(eps),
                                static_cast<const int64_t *>(ptr(pos)), ptr(cos_table), ptr(sin_table), n_pos, stream_of(dev)));
    return true;
}

// ---- between two linear layers of a block --------------------------------------------------------------------------
// Tensors that tensor operations would treat as nothing but their values, 16-byte aligned and one row behind another.
bool plain_rows(const Tensor &t, at::ScalarType dtype, const at::Device &dev, int64_t numel) {
    return t.defined() && t.scalar_type() == dtype && t.device() == dev && t.is_contiguous() && t.numel() == numel &&
           !at::isTensorSubclassLike(t) && !t._fw_grad(0).defined() && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
}
// Whether a mode on the torch-function stack looks at calls.  `with torch.device(...)` and torch.set_default_device put one there
// too, which only fills in the device of factory functions; the outputs here are allocated on their inputs' device.
bool function_modes() {
    if (!at::impl::torch_function_mode_enabled()) return false;
    using Tls = at::impl::PythonTorchFunctionTLS;
    static PyObject *device_context = nullptr;              // (under the GIL; no guard that an import could wait for)
    if (device_context == nullptr) device_context = py::object(py::module_::import("torch.utils._device").attr("DeviceContext")).release().ptr();
    for (int64_t i = 0; i < Tls::stack_len(); ++i)
        if (reinterpret_cast<PyObject *>(Py_TYPE(Tls::get_stack_at(i)->ptr(getPyInterpreter()))) != device_context) return true;
    return false;
}
bool watched() {
    return at::GradMode::is_enabled() || at::autocast::is_autocast_enabled(at::kCUDA) || torch::jit::tracer::isTracing() ||
           c10::impl::TorchDispatchModeTLS::any_modes_set() || function_modes();
}

// act(x W^T + bias), where the kernel measured faster than the library's product.  None: it did not, or this is no plain call.
std::optional<Tensor> linear(const Tensor &x, const Tensor &weight, const std::optional<Tensor> &bias, bool gelu) {
    if (watched() || !x.is_cuda() || at::isTensorSubclassLike(x) || x.dim() != 2 || x.numel() == 0 || weight.dim() != 2) return std::nullopt;
    const auto dtype = x.scalar_type();
    const int64_t rows = x.size(0), K = x.size(1), N = weight.size(0);
    const at::Device dev = x.device();
    const int act = gelu ? COME_ACT_GELU : COME_ACT_NONE;
    if ((dtype != at::kHalf && dtype != at::kBFloat16) || weight.size(1) != K || !abi.come_linear_is_faster(rows, K, N, act) ||
        !plain_rows(x, dtype, dev, rows * K) || !plain_rows(weight, dtype, dev, N * K) || (bias && !plain_rows(*bias, dtype, dev, N)))
        return std::nullopt;
    c10::DeviceGuard guard(dev);
    Tensor out = empty({rows, N}, dtype, dev);
    check(abi.come_linear(x.data_ptr(), weight.data_ptr(), bias ? bias->data_ptr() : nullptr, dtype_code(dtype), rows, K, N, act,
                          out.data_ptr(), stream_of(dev)));
    return out;
}

// x + scale * y and, where `norm`, its LayerNorm.  None: not a plain call (tensor operations do it then).
std::optional<std::tuple<Tensor, std::optional<Tensor>>> residual_norm(const Tensor &x, const Tensor &y, const Tensor &scale, bool norm,
                                                                       const std::optional<Tensor> &weight,
                                                                       const std::optional<Tensor> &bias, double eps) {
    if (watched() || !x.is_cuda() || at::isTensorSubclassLike(x) || x.dim() != 2 || x.numel() == 0 || y.sizes() != x.sizes()) return std::nullopt;
    const auto dtype = x.scalar_type();
    const int64_t rows = x.size(0), C = x.size(1), row_bytes = C * x.element_size();
    const at::Device dev = x.device();
    if ((dtype != at::kFloat && dtype != at::kHalf && dtype != at::kBFloat16) || row_bytes % 16 != 0 || row_bytes > 8192 ||
        !plain_rows(x, dtype, dev, rows * C) || !plain_rows(y, dtype, dev, rows * C) || !plain_rows(scale, dtype, dev, C) ||
        (weight && !plain_rows(*weight, dtype, dev, C)) || (bias && !plain_rows(*bias, dtype, dev, C)))
        return std::nullopt;
    c10::DeviceGuard guard(dev);
    Tensor sum = empty({rows, C}, dtype, dev);
    std::optional<Tensor> normed;
    if (norm) normed = empty({rows, C}, dtype, dev);
    check(abi.come_residual_norm(x.data_ptr(), y.data_ptr(), scale.data_ptr(), dtype_code(dtype), rows, C, rows, 0,
                                 weight ? weight->data_ptr() : nullptr, bias ? bias->data_ptr() : nullptr, static_cast<float>(eps),
                                 sum.data_ptr(), norm ? normed->data_ptr() : nullptr, stream_of(dev)));
    return std::make_tuple(sum, normed);
}

// A linear layer and the residual step behind it where few rows are worth cutting its sums into shares: those meet in the
// residual kernel.  None: they are not, or this is no plain call.
std::optional<std::tuple<Tensor, std::optional<Tensor>>> linear_residual_norm(const Tensor &a, const Tensor &w, const std::optional<Tensor> &b,
                                                                              const Tensor &x, const Tensor &scale, bool norm,
                                                                              const std::optional<Tensor> &weight,
                                                                              const std::optional<Tensor> &bias, double eps) {
    if (watched() || !a.is_cuda() || at::isTensorSubclassLike(a) || a.dim() != 2 || x.dim() != 2 || a.numel() == 0 || w.dim() != 2) return std::nullopt;
    const auto dtype = a.scalar_type();
    const at::Device dev = a.device();
    const int64_t rows = a.size(0), K = a.size(1), N = w.size(0);
    if ((dtype != at::kBFloat16 && dtype != at::kHalf) || w.size(1) != K || x.size(0) != rows || x.size(1) != N || N > 1024) return std::nullopt;
    const int64_t splits = abi.come_linear_splits(rows, K, N);
    if (splits < 2 || !plain_rows(a, dtype, dev, rows * K) || !plain_rows(w, dtype, dev, N * K) || (b && !plain_rows(*b, dtype, dev, N)) ||
        !plain_rows(x, dtype, dev, rows * N) || !plain_rows(scale, dtype, dev, N) || (weight && !plain_rows(*weight, dtype, dev, N)) ||
        (bias && !plain_rows(*bias, dtype, dev, N)))
        return std::nullopt;
    c10::DeviceGuard guard(dev);
    const hipStream_t stream = stream_of(dev);
    const int code = dtype_code(dtype);
    const Tensor partial = empty({splits, rows, N}, at::kFloat, dev);
    check(abi.come_linear_split(a.data_ptr(), w.data_ptr(), code, rows, K, N, static_cast<int>(splits), data<float>(partial), stream));
    Tensor sum = empty({rows, N}, dtype, dev);
    std::optional<Tensor> normed;
    if (norm) normed = empty({rows, N}, dtype, dev);
    check(abi.come_residual_norm_split(x.data_ptr(), data<float>(partial), static_cast<int>(splits), b ? b->data_ptr() : nullptr, scale.data_ptr(),
                                       code, rows, N, weight ? weight->data_ptr() : nullptr, bias ? bias->data_ptr() : nullptr,
                                       static_cast<float>(eps), sum.data_ptr(), norm ? normed->data_ptr() : nullptr, stream));
    return std::make_tuple(sum, normed);
}

// ---- a whole pre-norm block ------------------------------------------------------------------------------------------
// norm1 -> qkv -> q / k prologue -> attention -> proj -> residual, norm2 -> fc1, GELU -> fc2 -> residual (and norm1 of the block
// behind it): what harness.JaggedBlock does operator by operator, in one call.  A forward of one small frame is nothing but
// 48 such blocks being issued: 5.5 ms operator by operator, 4.7 in one call each (62 us of it the eight launches and their
// outputs); one of two frames, where the GPU has 6.4 ms to do, 6.6 and 6.5.  `fuse` false: LayerNorms and linear layers are
// the modules' own operations.  None: something is not plain, and nothing has been done.
struct Rows {                                                            // what the parameters are checked against
    at::ScalarType dtype;
    at::Device dev;
    bool ok(const Tensor &t, int64_t numel) const { return plain_rows(t, dtype, dev, numel); }
    bool ok(const std::optional<Tensor> &t, int64_t numel) const { return !t || ok(*t, numel); }
};

std::optional<std::tuple<Tensor, std::optional<Tensor>>> block(
    const Tensor &x, const std::optional<Tensor> &normed, const std::vector<std::optional<Tensor>> &params, const std::vector<double> &eps,
    int64_t heads, const Tensor &pos, const Tensor &cos_table, const Tensor &sin_table, int64_t n_pos, const Tensor &cu, int64_t max_seqlen,
    const std::optional<Tensor> &bias, double scale, int flags, bool fuse, bool has_next) {
    enum { kNorm1W, kNorm1B, kQkvW, kQkvB, kQW, kQB, kKW, kKB, kProjW, kProjB, kScale1, kNorm2W, kNorm2B, kFc1W, kFc1B, kFc2W, kFc2B, kScale2,
           kNextW, kNextB, kCount };
    if (watched() || params.size() != kCount || eps.size() != 4 || !x.is_cuda() || at::isTensorSubclassLike(x) || x.dim() != 2 || x.numel() == 0)
        return std::nullopt;
    const auto dtype = x.scalar_type();
    const at::Device dev = x.device();
    const int64_t P = x.size(0), C = x.size(1), D = heads > 0 ? C / heads : 0;
    for (const int i : {kQkvW, kProjW, kScale1, kFc1W, kFc2W, kScale2})
        if (!params[i]) return std::nullopt;
    const int64_t hidden = params[kFc1W]->numel() / C;
    const Rows rows{dtype, dev};
    if ((dtype != at::kBFloat16 && dtype != at::kHalf) || D * heads != C || D != 64 || C * 2 > 8192 ||
        max_seqlen < 2 || !rows.ok(x, P * C) || !rows.ok(normed, P * C) || !rows.ok(params[kNorm1W], C) || !rows.ok(params[kNorm1B], C) ||
        !rows.ok(params[kQkvW], 3 * C * C) || !rows.ok(params[kQkvB], 3 * C) || !rows.ok(params[kQW], D) || !rows.ok(params[kQB], D) ||
        !rows.ok(params[kKW], D) || !rows.ok(params[kKB], D) || !rows.ok(params[kProjW], C * C) || !rows.ok(params[kProjB], C) ||
        !rows.ok(params[kScale1], C) || !rows.ok(params[kNorm2W], C) || !rows.ok(params[kNorm2B], C) || !rows.ok(params[kFc1W], hidden * C) ||
        !rows.ok(params[kFc1B], hidden) || !rows.ok(params[kFc2W], hidden * C) || !rows.ok(params[kFc2B], C) || !rows.ok(params[kScale2], C) ||
        !rows.ok(params[kNextW], C) || !rows.ok(params[kNextB], C) || !rows.ok(cos_table, n_pos * D / 4) || !rows.ok(sin_table, n_pos * D / 4) ||
        !plain_rows(pos, at::kLong, dev, 2 * P) || !cu.is_cuda() || cu.scalar_type() != at::kInt || cu.dim() != 1 || !cu.is_contiguous() ||
        cu.numel() < 2 || cu.device() != dev || (bias && (!rows.ok(*bias, P) || bias->dim() != 1)))
        return std::nullopt;
    for (const int i : {kQkvW, kProjW, kFc1W, kFc2W})
        if (params[i]->dim() != 2 || params[i]->size(1) != (i == kFc2W ? hidden : C)) return std::nullopt;
    c10::DeviceGuard guard(dev);
    auto product = [&](const Tensor &a, int w, int b, bool gelu) {
        if (fuse)
            if (auto y = linear(a, *params[w], params[b], gelu)) return *y;
        const Tensor y = at::linear(a, *params[w], params[b]);
        return gelu ? at::gelu(y) : y;
    };
    auto norm = [&](const Tensor &a, int w, int b, double e) { return at::layer_norm(a, {C}, params[w], params[b], e); };
    // a + scale * (linear layer of h), and its norm
    auto residual = [&](const Tensor &a, const Tensor &h, int lw, int lb, int s, bool with_norm, int w, int b, double e) {
        if (fuse)
            if (auto r = linear_residual_norm(h, *params[lw], params[lb], a, *params[s], with_norm, params[w], params[b], e)) return *r;
        auto r = residual_norm(a, product(h, lw, lb, false), *params[s], with_norm && fuse, params[w], params[b], e).value();
        if (with_norm && !fuse) std::get<1>(r) = norm(std::get<0>(r), w, b, e);
        return r;
    };
    const Tensor qkv = product(normed ? *normed : norm(x, kNorm1W, kNorm1B, eps[0]), kQkvW, kQkvB, false).view({P, 3, heads, D});
    qk_norm_rope(qkv, false, true, eps[1], params[kQW], params[kQB], params[kKW], params[kKB], pos, cos_table, sin_table, n_pos);
    const Tensor o = attention(qkv, cu, max_seqlen, bias, scale, flags).value().view({P, C});
    const auto [x1, h1] = residual(x, o, kProjW, kProjB, kScale1, true, kNorm2W, kNorm2B, eps[2]);
    const Tensor a = product(*h1, kFc1W, kFc1B, true);
    return residual(x1, a, kFc2W, kFc2B, kScale2, has_next, kNextW, kNextB, eps[3]);
}

// LayerNorm over the last dimension of x [groups, n, C], whose groups may lie apart; the result is contiguous.  None: as above.
std::optional<Tensor> layer_norm_groups(const Tensor &x, const std::optional<Tensor> &weight, const std::optional<Tensor> &bias, double eps) {
    if (watched() || !x.is_cuda() || at::isTensorSubclassLike(x) || x._fw_grad(0).defined() || x.dim() != 3 || x.numel() == 0) return std::nullopt;
    const auto dtype = x.scalar_type();
    const int64_t G = x.size(0), n = x.size(1), C = x.size(2), size = x.element_size(), row_bytes = C * size;
    const at::Device dev = x.device();
    if ((dtype != at::kFloat && dtype != at::kHalf && dtype != at::kBFloat16) || row_bytes % 16 != 0 || row_bytes > 8192 ||
        x.stride(2) != 1 || (n > 1 && x.stride(1) != C) || (G > 1 && (x.stride(0) < n * C || x.stride(0) * size % 16 != 0)) ||
        reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 != 0 || (weight && !plain_rows(*weight, dtype, dev, C)) ||
        (bias && !plain_rows(*bias, dtype, dev, C)))
        return std::nullopt;
    c10::DeviceGuard guard(dev);
    Tensor out = empty({G, n, C}, dtype, dev);
    check(abi.come_residual_norm(x.data_ptr(), nullptr, nullptr, dtype_code(dtype), G * n, C, n, x.stride(0),
                                 weight ? weight->data_ptr() : nullptr, bias ? bias->data_ptr() : nullptr, static_cast<float>(eps),
                                 nullptr, out.data_ptr(), stream_of(dev)));
    return out;
}

// ---- suffix operators ----------------------------------------------------------------------------------------------
std::tuple<Tensor, Tensor, Tensor> add_suffix(const Tensor &tokens, const Tensor &weight, const Tensor &offset, const Tensor &suffix) {
    const at::Device dev = tokens.device();
    c10::DeviceGuard guard(dev);
    const int64_t M = offset.size(0) - 1, T = suffix.size(1), C = suffix.size(2), P = tokens.size(1);
    const Tensor t = tokens.contiguous(), w = weight.to(dev, at::kFloat).contiguous(), o = offset.to(dev, at::kLong).contiguous(),
                 s = suffix.to(dev, tokens.scalar_type()).contiguous();
    Tensor out = empty({1, P + M * T, C}, tokens.scalar_type(), dev), out_w = empty({P + M * T}, at::kFloat, dev),
           out_o = empty({M + 1}, at::kLong, dev);
    check(abi.come_jagged_add_suffix(t.data_ptr(), data<float>(w), dtype_code(t.scalar_type()), P, C, data<int64_t>(o), M, s.data_ptr(),
                                     T, out.data_ptr(), data<float>(out_w), data<int64_t>(out_o), stream_of(dev)));
    return {out, out_w.to(weight.scalar_type()), out_o.to(offset.scalar_type())};
}

// None: some segment is shorter than the suffix
py::object split_suffix(const Tensor &tokens, const Tensor &weight, const Tensor &offset, int64_t T) {
    const at::Device dev = tokens.device();
    c10::DeviceGuard guard(dev);
    const int64_t M = offset.size(0) - 1, C = tokens.size(2), P = tokens.size(1);
    const Tensor t = tokens.contiguous(), w = weight.to(dev, at::kFloat).contiguous(), o = offset.to(dev, at::kLong).contiguous();
    Tensor out = empty({1, P - M * T, C}, tokens.scalar_type(), dev), out_w = empty({P - M * T}, at::kFloat, dev),
           out_o = empty({M + 1}, at::kLong, dev), suffix = empty({M, T, C}, tokens.scalar_type(), dev);
    const hipStream_t stream = stream_of(dev);
    Post verdict(stream);
    check(abi.come_jagged_split_suffix_post(t.data_ptr(), data<float>(w), dtype_code(t.scalar_type()), P, C, data<int64_t>(o), M, T,
                                            out.data_ptr(), data<float>(out_w), data<int64_t>(out_o), suffix.data_ptr(),
                                            verdict.word(), verdict.tag(), stream));
    verdict.launched();
    uint32_t too_short = 0;
    if (!verdict.wait(too_short))                                        // no word to post to: read the lengths back
        too_short = M > 0 && (o.narrow(0, 1, M) - o.narrow(0, 0, M)).min().item<int64_t>() < T;
    if (too_short) return py::none();
    return py::make_tuple(out, out_w.to(weight.scalar_type()), out_o.to(offset.scalar_type()), suffix);
}

}  // namespace

PYBIND11_MODULE(_come_host, m) {
    using torch::wrap_pybind_function;
    m.def("bind", &bind);
    m.def("select_mask", wrap_pybind_function(&select_mask));
    m.def("select_merge_2d", wrap_pybind_function(&select_merge_2d));
    m.def("merge_2d", wrap_pybind_function(&merge_2d));
    m.def("merge_1d", wrap_pybind_function(&merge_1d));
    m.def("merge_2d_flat", wrap_pybind_function(&merge_2d_flat));
    m.def("split", wrap_pybind_function(&split));
    m.def("attention", wrap_pybind_function(&attention));
    m.def("qk_norm_rope", wrap_pybind_function(&qk_norm_rope));
    m.def("block", wrap_pybind_function(&block));
    m.def("linear_residual_norm", wrap_pybind_function(&linear_residual_norm));
    m.def("linear", wrap_pybind_function(&linear));
    m.def("residual_norm", wrap_pybind_function(&residual_norm));
    m.def("layer_norm_groups", wrap_pybind_function(&layer_norm_groups));
    m.def("add_suffix", wrap_pybind_function(&add_suffix));
    m.def("split_suffix", wrap_pybind_function(&split_suffix));
}

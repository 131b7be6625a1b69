// The host side of the operators: argument checks, output allocation and the calls into libcome_hip.so, in native code.
//
// A merge or unmerge of one frame is 3 - 5 us of kernel, so what a call costs is the host path in front of the launch:
// through Python and ctypes a split took 11.4 us (about twenty interpreter-level tensor calls and a 20-argument foreign
// call); here it is one call that allocates through the caching allocator directly and launches.  The C ABI of
// libcome_hip.so stays the product's boundary: this module looks its functions up in the library the Python binding has
// loaded (bind) and knows nothing of its kernels.
//
// The packed row count of a merge decides the shape of its outputs, so it has to reach the host.  The plan kernels store
// it into pinned host memory (a Mailbox slot) while they run; the host polls that word.  For a plan made from fp32
// confidences by rank the count is known in advance unless window means tie at the threshold: the merge is then launched
// at once with outputs of the expected size and the posted count confirms it afterwards.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/csrc/utils/pybind.h>

#include <ATen/ATen.h>
#include <ATen/TensorSubclassLikeUtils.h>
#include <ATen/autocast_mode.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/DeviceGuard.h>
#include <dlfcn.h>
#include <hip/hip_runtime_api.h>

#include <atomic>
#include <chrono>
#include <cmath>
#include <memory>
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
    F(come_last_error) F(come_merge_plan_post) F(come_token_merge_wide) F(come_token_split) F(come_token_split_pair) \
    F(come_select_plan_post) F(come_attn_work_bytes)                \
    F(come_attn_varlen_fwd_ws) F(come_qk_norm_rope) F(come_jagged_add_suffix)            \
    F(come_jagged_split_suffix_post) F(come_residual_norm)
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
// kernel still running can write into a word that somebody else waits for.  A plan that dies unread leaves its word on
// the waiting list until the post has arrived.  Without a free word (512 plans alive) callers read the count back instead.
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

// ---- merge plan -------------------------------------------------------------------------------------------------
// From a merge mask to packed positions: what both merges of a pass (tokens and positions) need, made once.
class MergePlan {
public:
    int64_t rows = 0, groups = 0, start = 0, group_size = 0, tail = 0;
    int64_t expected = -1;                              // packed rows if no two window means tie at the threshold, -1: unknown
    Tensor offsets, prefix;                             // int32 [rows + 1], [rows, groups]
    // the mask the plan was made from: storage address and version, so that a mask that has been written to since is
    // planned again
    const void *mask_ptr = nullptr;
    uint32_t mask_version = 0;
    bool versioned = false;

    ~MergePlan() { mailbox().give_back(slot_); }

    void allocate(const at::Device &dev, int64_t rows_, int64_t groups_, int64_t start_, int64_t group_size_, int64_t tail_) {
        rows = rows_;
        groups = groups_;
        start = start_;
        group_size = group_size_;
        tail = tail_;
        // (the prefix starts at a multiple of 16 bytes)
        const int64_t n_off = (rows + 1 + 3) / 4 * 4;
        const Tensor both = empty({n_off + std::max<int64_t>(rows * groups, 1)}, at::kInt, dev);
        offsets = both.narrow(0, 0, rows + 1);
        prefix_ptr_ = data<int32_t>(both) + n_off;
        device_ = dev;
        stream_ = stream_of(dev);
        slot_ = mailbox().take();
    }
    int32_t *prefix_ptr() const { return prefix_ptr_; }
    uint64_t *post() const { return mailbox().word(slot_); }
    uint32_t tag() const { return slot_.tag; }
    hipStream_t stream() const { return stream_; }
    void launch_failed() {
        mailbox().give_back_unused(slot_);
        slot_ = Mailbox::Slot();
    }
    void of_mask(const Tensor &mask) {
        versioned = !mask.is_inference();
        mask_ptr = mask.data_ptr();
        mask_version = versioned ? mask._version() : 0;
    }
    bool made_from(const Tensor &mask, int64_t start_, int64_t group_size_, int64_t tail_) const {
        return versioned && !mask.is_inference() && mask.data_ptr() == mask_ptr && mask._version() == mask_version &&
               mask.dim() == 2 && mask.size(0) == rows && mask.size(1) == groups && start == start_ &&
               group_size == group_size_ && tail == tail_ && mask.device() == device_ &&
               stream_of(device_) == stream_;              // (a plan's buffers are ordered with the stream that made them)
    }
    // Packed rows: posted by the plan's launch, read back from the offsets where there was no word for it.
    int64_t packed_rows() {
        if (packed_ >= 0) return packed_;
        if (rows == 0) return packed_ = 0;
        uint32_t v = 0;
        if (mailbox().wait(slot_, stream_, v)) return packed_ = v;
        c10::DeviceGuard guard(device_);
        return packed_ = offsets.select(0, rows).item<int32_t>();
    }

private:
    Mailbox::Slot slot_;
    int32_t *prefix_ptr_ = nullptr;
    at::Device device_ = at::kCPU;
    hipStream_t stream_ = nullptr;
    int64_t packed_ = -1;
};

// confidence -> (mask, plan).  The grid holds at least one full window.
std::tuple<Tensor, std::shared_ptr<MergePlan>> select_plan(const Tensor &confidence, int64_t batch, int64_t rows, int64_t H,
                                                           int64_t W, int64_t gh, int64_t gw, double threshold, int mode,
                                                           int64_t start) {
    require(confidence.is_cuda(), "conf must be on CUDA");
    const auto dtype = confidence.scalar_type();
    require(dtype == at::kBFloat16 || dtype == at::kFloat, "conf must be bfloat16 or float32");
    const Tensor conf = confidence.contiguous();
    const at::Device dev = conf.device();
    c10::DeviceGuard guard(dev);
    const int64_t M = (H / gh) * (W / gw), G = gh * gw;
    auto plan = std::make_shared<MergePlan>();
    Tensor mask = empty({rows, M}, at::kBool, dev);
    plan->allocate(dev, rows, M, start, G, H * W - M * G);
    const int64_t n = rows / batch * M;
    Tensor means;
    if (n > 16384) means = empty({batch * n}, at::kFloat, dev);          // fewer keys stay in the workgroup's LDS
    const int status = abi.come_select_plan_post(
        conf.data_ptr(), dtype_code(dtype), batch, rows / batch, H, W, gh, gw, mode, static_cast<float>(threshold), start,
        means.defined() ? data<float>(means) : nullptr, data<uint8_t>(mask), data<int32_t>(plan->offsets), plan->prefix_ptr(),
        nullptr, 0, plan->post(), plan->tag(), plan->stream());
    if (status != COME_OK) {
        plan->launch_failed();
        check(status);
    }
    plan->of_mask(mask);
    if (mode == 0 && dtype == at::kFloat) {
        // q = quantile(means, threshold): with distinct means floor(rank) + 1 of them lie below it, floor(rank) where the
        // rank is a whole number (q is then one of the means).  bf16 means tie all the time: not expected, waited for.
        const float rank = static_cast<float>(threshold) * static_cast<float>(n - 1);
        const float low = std::floor(rank);
        const int64_t merged = static_cast<int64_t>(low) + (rank > low ? 1 : 0);
        plan->expected = rows * (start + H * W) - batch * merged * (G - 1);
    }
    return {mask, plan};
}

std::shared_ptr<MergePlan> plan_of_mask(const Tensor &mask, int64_t start, int64_t G, int64_t tail) {
    auto plan = std::make_shared<MergePlan>();
    plan->allocate(mask.device(), mask.size(0), mask.size(1), start, G, tail);
    const int status = abi.come_merge_plan_post(mask.numel() > 0 ? data<uint8_t>(mask) : nullptr, plan->rows, plan->groups, start, G,
                                                tail, data<int32_t>(plan->offsets), plan->prefix_ptr(), plan->post(),
                                                plan->tag(), plan->stream());
    if (status != COME_OK) {
        plan->launch_failed();
        check(status);
    }
    return plan;
}

struct Merged {
    Tensor out, offsets32, offsets64, index_map, counts;
};

// tokens [rows, n_tok, C] (or [B, S, n_tok, C]), contiguous; packed: shape of the packed tensor [1, P, C] or [P, C]
Merged merge(const Tensor &tokens, int64_t rows, int64_t n_tok, int64_t C, int64_t start, int64_t gh, int64_t gw, int64_t H,
             int64_t W, const Tensor &mask, std::shared_ptr<MergePlan> plan, at::ScalarType index_dtype,
             at::ScalarType count_dtype, bool wide, bool lead) {
    const at::Device dev = tokens.device();
    const int code = dtype_code(tokens.scalar_type());
    const int64_t M = (H / gh) * (W / gw), G = gh * gw, tail = H * W - M * G;
    if (!plan || !plan->made_from(mask, start, G, tail)) plan = plan_of_mask(mask, start, G, tail);
    Merged m;
    m.offsets32 = plan->offsets;
    m.index_map = empty({rows * n_tok}, index_dtype, dev);
    if (wide) m.offsets64 = empty({rows + 1}, at::kLong, dev);
    const hipStream_t stream = stream_of(dev);
    auto launch = [&](int64_t P) {
        m.out = lead ? empty({1, P, C}, tokens.scalar_type(), dev) : empty({P, C}, tokens.scalar_type(), dev);
        m.counts = empty({P}, count_dtype, dev);
        void *index = m.index_map.data_ptr(), *counts = m.counts.data_ptr();
        check(abi.come_token_merge_wide(
            tokens.data_ptr(), code, rows, n_tok, C, start, gh, gw, H, W, mask.numel() > 0 ? data<uint8_t>(mask) : nullptr,
            data<int32_t>(plan->offsets), plan->prefix_ptr(), m.out.data_ptr(), P,
            index_dtype == at::kLong ? static_cast<int64_t *>(index) : nullptr,
            index_dtype == at::kInt ? static_cast<int32_t *>(index) : nullptr,
            count_dtype == at::kFloat ? static_cast<float *>(counts) : nullptr,
            count_dtype == at::kInt ? static_cast<int32_t *>(counts) : nullptr, wide ? data<int64_t>(m.offsets64) : nullptr, stream));
    };
    if (plan->expected > 0 && rows > 0) {
        launch(plan->expected);                          // (rows beyond the outputs are not written)
        const int64_t P = plan->packed_rows();
        if (P != plan->expected) launch(plan->expected = P);          // means tied at the threshold
    } else {
        launch(plan->packed_rows());
    }
    if (wide && (rows == 0 || n_tok == 0)) m.offsets64 = plan->offsets.to(at::kLong);      // nothing was launched
    return m;
}

// ---- token merger entry points.  None: the arguments are not what the operator takes; the caller's checks say why. ----
py::object merge_2d(const Tensor &tokens, int64_t start, int64_t gh, int64_t gw, int64_t H, int64_t W, const Tensor &mask,
                    bool allow_remainder, std::shared_ptr<MergePlan> plan) {
    const int64_t d = tokens.dim();
    if (d != 3 && d != 4) return py::none();
    const int64_t rows = d == 4 ? tokens.size(0) * tokens.size(1) : tokens.size(0), n_tok = tokens.size(d - 2), C = tokens.size(d - 1);
    if (!tokens.is_cuda() || !mask.is_cuda() || mask.scalar_type() != at::kBool || mask.dim() != 2 || start < 0 || gh <= 0 || gw <= 0 ||
        H < 0 || W < 0 || (!allow_remainder && (H % gh != 0 || W % gw != 0)) || mask.size(0) != rows || n_tok != start + H * W ||
        mask.size(1) != (H / gh) * (W / gw) || mask.device() != tokens.device())
        return py::none();
    c10::DeviceGuard guard(tokens.device());
    const Merged m = merge(tokens.contiguous(), rows, n_tok, C, start, gh, gw, H, W, mask.contiguous(), std::move(plan), at::kLong,
                           at::kFloat, true, true);
    return py::make_tuple(m.out, m.counts, m.offsets64, m.index_map);
}

py::object merge_1d(const Tensor &tokens, int64_t start, int64_t G, const Tensor &mask, bool wide) {
    if (tokens.dim() != 3 || mask.dim() != 2 || !tokens.is_cuda() || !mask.is_cuda() || mask.scalar_type() != at::kBool || start < 0 ||
        G <= 0 || mask.size(0) != tokens.size(0) || tokens.size(1) != start + mask.size(1) * G || mask.device() != tokens.device())
        return py::none();
    c10::DeviceGuard guard(tokens.device());
    const int64_t M = mask.size(1);
    const Merged m = merge(tokens.contiguous(), tokens.size(0), tokens.size(1), tokens.size(2), start, 1, G, M > 0 ? 1 : 0, M * G,
                           mask.contiguous(), nullptr, at::kLong, at::kFloat, wide, wide);
    return py::make_tuple(m.out, wide ? m.offsets64 : m.offsets32, m.index_map, m.counts);
}

// the operator with the caller's index and count types: (out [P, C], offsets int32, index_map, counts)
py::tuple merge_2d_flat(const Tensor &tokens, int64_t start, int64_t gh, int64_t gw, int64_t H, int64_t W, const Tensor &mask,
                        bool index_64, bool count_float, std::shared_ptr<MergePlan> plan) {
    c10::DeviceGuard guard(tokens.device());
    const Merged m = merge(tokens.contiguous(), tokens.size(0), tokens.size(1), tokens.size(2), start, gh, gw, H, W, mask.contiguous(),
                           std::move(plan), index_64 ? at::kLong : at::kInt, count_float ? at::kFloat : at::kInt, false, false);
    return py::make_tuple(m.out, m.offsets32, m.index_map, m.counts);
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
bool watched() { return at::GradMode::is_enabled() || at::autocast::is_autocast_enabled(at::kCUDA) || torch::jit::tracer::isTracing(); }

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
    const Mailbox::Slot slot = mailbox().take();
    const int status = abi.come_jagged_split_suffix_post(t.data_ptr(), data<float>(w), dtype_code(t.scalar_type()), P, C, data<int64_t>(o),
                                                         M, T, out.data_ptr(), data<float>(out_w), data<int64_t>(out_o),
                                                         suffix.data_ptr(), mailbox().word(slot), slot.tag, stream);
    if (status != COME_OK) {
        mailbox().give_back_unused(slot);
        check(status);
    }
    uint32_t too_short = 0;
    const bool posted = mailbox().wait(slot, stream, too_short);
    mailbox().give_back(slot);
    if (!posted)                                        // no word to post to: read the lengths back
        too_short = M > 0 && (o.narrow(0, 1, M) - o.narrow(0, 0, M)).min().item<int64_t>() < T;
    if (too_short) return py::none();
    return py::make_tuple(out, out_w.to(weight.scalar_type()), out_o.to(offset.scalar_type()), suffix);
}

}  // namespace

PYBIND11_MODULE(_come_host, m) {
    using torch::wrap_pybind_function;
    m.def("bind", &bind);
    // A copied or saved mask leaves its plan behind (device buffers, a word that a kernel posts to): an empty OrderedDict,
    // which every loader knows, stands in its place, and a merge with that mask plans again.
    py::class_<MergePlan, std::shared_ptr<MergePlan>>(m, "MergePlan")
        .def("packed_rows", wrap_pybind_function(&MergePlan::packed_rows))
        .def("__reduce_ex__", [](const MergePlan &, int) {
            return py::make_tuple(py::module_::import("collections").attr("OrderedDict"), py::tuple());
        });
    m.def("select_plan", wrap_pybind_function(&select_plan));
    m.def("merge_2d", wrap_pybind_function(&merge_2d));
    m.def("merge_1d", wrap_pybind_function(&merge_1d));
    m.def("merge_2d_flat", wrap_pybind_function(&merge_2d_flat));
    m.def("split", wrap_pybind_function(&split));
    m.def("attention", wrap_pybind_function(&attention));
    m.def("qk_norm_rope", wrap_pybind_function(&qk_norm_rope));
    m.def("residual_norm", wrap_pybind_function(&residual_norm));
    m.def("layer_norm_groups", wrap_pybind_function(&layer_norm_groups));
    m.def("add_suffix", wrap_pybind_function(&add_suffix));
    m.def("split_suffix", wrap_pybind_function(&split_suffix));
}

// The package's operators and the layer's forward and backward passes on torch tensors: what a call allocates, checks and launches,
// as native code.  A training step of a small layer is launches only (eight kernels of 2 to 8 us each), so the time that the host
// takes per launch is what the step takes: forward and backward of a 256 x 1024 x 1024 layer in fp32 were 220 us of Python, autograd
// and ctypes around 43 us of kernels.  Here one call takes its intermediate codes and scales from one allocation, quantizes X and W
// in one launch, and the backward pass runs on autograd's own thread without the interpreter.
//
// Replaces triton_functions.py:142-168, :221-233, :492-500 (the launchers) and block_linear.py:69-112 (the autograd function).
#include <Python.h>

#include <cstring>

#include <ATen/ATen.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_variable.h>

#include "bi8_internal.h"

namespace {

using at::ScalarType;
using at::Tensor;

// The library's refusals, raised as the package's Bi8Error; its operand checks, raised as AssertionError like the reference's asserts.
struct Bi8Failure : std::runtime_error {
    using std::runtime_error::runtime_error;
};
struct OperandError : std::runtime_error {
    using std::runtime_error::runtime_error;
};
struct TypeFailure : std::runtime_error {
    using std::runtime_error::runtime_error;
};

void check(int rc, const char *what) {
    if (rc != BI8_OK) throw Bi8Failure(std::string(what) + " failed: " + bi8_strerror(rc) + " (code " + std::to_string(rc) + ")");
}
void require(bool ok, const char *what) {
    if (!ok) throw OperandError(what);
}

int dtype_code(ScalarType t) { return t == at::kFloat ? BI8_F32 : t == at::kBFloat16 ? BI8_BF16 : t == at::kHalf ? BI8_F16 : -1; }
int float_code(const Tensor &x) {
    const int c = dtype_code(x.scalar_type());
    if (c < 0) throw TypeFailure(std::string("unsupported dtype ") + c10::toString(x.scalar_type()) + ": expected float32, bfloat16 or float16");
    return c;
}
void *stream_of(const Tensor &t) { return (void *)c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
Tensor empty(at::IntArrayRef size, ScalarType type, const Tensor &like) { return Tensor(at::detail::empty_cuda(size, type, like.device(), std::nullopt)); }
int64_t up(int64_t n, int64_t to) { return (n + to - 1) / to * to; }
int64_t ceil_div(int64_t n, int64_t d) { return (n + d - 1) / d; }

// a 2-D tensor whose rows are contiguous (leading dimension = stride(0)): x itself where it is one
Tensor rows_of(const Tensor &x) {
    if (x.is_contiguous()) return x;
    if (x.numel() != 0 && (x.stride(1) != 1 || (x.size(0) > 1 && x.stride(0) < x.size(1)))) return x.contiguous();
    return x;
}
int64_t ld_of(const Tensor &x) { return x.size(0) > 1 ? x.stride(0) : std::max<int64_t>(x.size(1), 1); }
// [..., K] -> [rows, K]
Tensor matrix_of(const Tensor &x) {
    if (x.dim() == 2) return rows_of(x);
    const int64_t k = x.size(-1);
    int64_t m = 1;
    for (int64_t d = 0; d + 1 < x.dim(); ++d) m *= x.size(d);
    return rows_of(x.reshape({m, k}));
}
std::vector<int64_t> with_last(const Tensor &x, int64_t n) {
    std::vector<int64_t> s(x.sizes().begin(), x.sizes().end());
    s.back() = n;
    return s;
}
bool fast_block(int64_t block) { return block == 32 || block == 64 || block == 128; }

// Scales are kept in SHARED_EXP_TORCH_TYPE (triton_functions.py:216, :227) and multiplied as fp32.
Tensor scales_out(const Tensor &s, ScalarType type) { return type == at::kFloat ? s : s.to(type); }
Tensor scales_in(const Tensor &s) { return (s.scalar_type() == at::kFloat ? s : s.to(at::kFloat)).contiguous(); }

struct Bias {
    Tensor held;
    const void *ptr = nullptr;
    int code = 0;
    Bias(const Tensor &b, int64_t n) {
        if (!b.defined()) return;
        require(b.is_cuda() && b.numel() == n, "bias must be a device tensor of one element per output column");
        held = (dtype_code(b.scalar_type()) < 0 ? b.to(at::kFloat) : b).contiguous();
        ptr = held.data_ptr();
        code = dtype_code(held.scalar_type());
    }
};

// ---- operators ------------------------------------------------------------------------------------------------------
std::pair<Tensor, Tensor> quantize_rowwise(const Tensor &x_in, int64_t block, ScalarType scale_type) {
    const int code = float_code(x_in);
    const Tensor x = rows_of(x_in);
    const int64_t m = x.size(0), k = x.size(1);
    c10::DeviceGuard guard(x.device());
    Tensor q = empty({m, k}, at::kChar, x), s = empty({ceil_div(k, block), m}, at::kFloat, x);
    check(bi8_quantize_rowwise(x.data_ptr(), code, (int8_t *)q.data_ptr(), (float *)s.data_ptr(), m, k, ld_of(x), std::max<int64_t>(k, 1), (int)block, stream_of(x)),
          "bi8_quantize_rowwise");
    return {q, scales_out(s, scale_type)};
}

std::pair<Tensor, Tensor> quantize_transposed(const Tensor &x_in, int64_t block, ScalarType scale_type) {
    const int code = float_code(x_in);
    const Tensor x = rows_of(x_in);
    const int64_t r = x.size(0), c = x.size(1);
    c10::DeviceGuard guard(x.device());
    Tensor q = empty({c, r}, at::kChar, x), s = empty({ceil_div(r, block), c}, at::kFloat, x);
    check(bi8_quantize_transposed(x.data_ptr(), code, (int8_t *)q.data_ptr(), (float *)s.data_ptr(), r, c, ld_of(x), std::max<int64_t>(r, 1), (int)block, stream_of(x)),
          "bi8_quantize_transposed");
    return {q, scales_out(s, scale_type)};
}

Tensor dequantize(const Tensor &q_in, const Tensor &state, int64_t block, ScalarType out_type) {
    require(q_in.scalar_type() == at::kChar, "codes must be int8");
    require(state.is_cuda(), "scales must be device tensors");
    const int64_t m = q_in.size(0), k = q_in.size(1);
    require(state.dim() == 2 && state.size(0) == ceil_div(k, block) && state.size(1) == m, "scale shape must be [ceil(K/block), M]");
    const Tensor q = rows_of(q_in), s = scales_in(state);
    c10::DeviceGuard guard(q.device());
    Tensor out = empty({m, k}, out_type, q);
    check(bi8_dequantize_rowwise((const int8_t *)q.data_ptr(), (const float *)s.data_ptr(), out.data_ptr(), float_code(out), m, k, ld_of(q), std::max<int64_t>(k, 1),
                                 (int)block, stream_of(q)),
          "bi8_dequantize_rowwise");
    return out;
}

// The GEMM on operands that need no preparation: codes [M,K] and [N,kw] with their scales, kw = K or K padded to a multiple of 128 in A.
int gemm_raw(const int8_t *a, const float *sa, int64_t lda, const int8_t *w, const float *sw, int64_t ldw, const Bias &bias, void *c, int c_code, int64_t M, int64_t N,
             int64_t K, int64_t kw, int64_t block, void *ws, int64_t ws_bytes, void *stream) {
    return bi8x_gemm(a, w, sa, sw, bias.ptr, bias.code, c, c_code, M, N, K, kw, lda, ldw, std::max<int64_t>(N, 1), (int)block, ws, ws_bytes, stream);
}
// Scratch bytes that the split of K wants (up to 16 rows at blocks 64 and 128 run one-pass kernels whatever they are given).
int64_t scratch_for(int64_t M, int64_t N, int64_t K, int64_t block) { return M <= 16 && block != 32 ? 0 : bi8_gemm_workspace_bytes(M, N, K, (int)block); }

// The last row's 16-byte chunk that holds its last codes lies inside w's storage (a range-checked load gives zeros for a dword that
// only partly lies in the range, so the range given to the kernels is whole chunks; w's rows are 16-byte aligned).
bool whole_chunks(const Tensor &w, int64_t contraction) {
    return (int64_t)w.storage().nbytes() >= w.storage_offset() + (w.size(0) - 1) * ld_of(w) + up(contraction, 16);
}
// M*N*K below which the general kernel is as quick as a padded copy
constexpr int64_t kPadMinWork = 1 << 22;
bool small_product(int64_t M, int64_t N, int64_t K) { return (double)M * (double)N * (double)K < (double)kPadMinWork; }
// Whether the layer multiplies codes padded along a contraction of K.  Small products with a ragged contraction stay with the general
// kernel, as the operator's do: the tiled kernels round the column scales to 22 bits (twice its fp32 error in the 2-norm) and make
// an infinite one NaN.  The few-row kernels take the scales as they are, so products that run on those are padded whatever the size.
bool pad_contraction(int64_t M, int64_t N, int64_t K, int64_t block) {
    const int64_t kp = up(K, 128);
    return kp == K || !small_product(M, N, K) || std::strncmp(bi8_gemm_kernel_name(M, N, kp, kp, kp, (int)block, scratch_for(M, N, kp, block)), "gemv_", 5) == 0;
}

// a [M,K] codes, w [N,K] codes (both with contiguous rows), any block size and alignment.
//  * A K-block of 256, 512, ... codes is two, four, ... runs of 128 codes that share their scales: with every scale row repeated
//    block/128 times the GEMM runs at block 128 on the MFMA kernels, where the library itself has only its general kernel for such
//    blocks (~40x slower).  (The reference's kernel takes any power of two as its BLOCK_K, triton_functions.py:30, :43-56.)
//  * The tiled kernels want K to be a multiple of 128 and 16-byte aligned operand rows; a contraction like the GPT-2 vocabulary (50257)
//    would fall to the general kernel.  Zero codes add nothing to any block partial, so A is copied once into rows padded with zero
//    codes up to the next multiple of 128 (and its scales with zero rows if that adds K-blocks); W too where its rows are not 16-byte
//    aligned or the block is 32, which the kernels that read W through range-checked buffers do not serve.
// `scratch`: memory that the split of K may use, instead of an allocation of its own.
Tensor gemm(Tensor a, Tensor w, Tensor sx, Tensor sw, const Tensor &bias_in, int64_t block, ScalarType out_type, const Tensor &scratch = Tensor()) {
    const int64_t M = a.size(0), N = w.size(0);
    int64_t K = a.size(1);
    require(sx.is_cuda() && sw.is_cuda(), "scales must be device tensors");
    require(sx.dim() == 2 && sw.dim() == 2 && sx.size(0) == ceil_div(K, block) && sx.size(1) == M && sw.size(0) == sx.size(0) && sw.size(1) == N,
            "scale shapes must be [ceil(K/block), rows]");
    c10::DeviceGuard guard(a.device());
    sx = scales_in(sx);
    sw = scales_in(sw);
    const bool worth = K > 0 && !small_product(M, N, K);
    if (block > 128 && (block & (block - 1)) == 0 && worth) {
        sx = sx.repeat_interleave(block / 128, 0).slice(0, 0, ceil_div(K, 128)).contiguous();
        sw = sw.repeat_interleave(block / 128, 0).slice(0, 0, ceil_div(K, 128)).contiguous();
        block = 128;
    }
    int64_t kw = K;
    auto unaligned = [](const Tensor &t) { return ld_of(t) % 16 != 0 || (uintptr_t)t.data_ptr() % 16 != 0; };
    if (fast_block(block) && worth && (K % 128 != 0 || unaligned(a) || unaligned(w))) {
        const int64_t kp = up(K, 128), extra = kp / block - sx.size(0);
        const bool pad_w = unaligned(w) || (block == 32 && kp != K) || !whole_chunks(w, K);
        if (kp != K || unaligned(a)) a = at::constant_pad_nd(a, {0, kp - K});
        if (extra > 0) sx = at::constant_pad_nd(sx, {0, 0, 0, extra});
        if (pad_w) {
            w = at::constant_pad_nd(w, {0, kp - K});
            if (extra > 0) sw = at::constant_pad_nd(sw, {0, 0, 0, extra});
            kw = kp;
        } else {
            kw = up(K, 16);
        }
        K = kp;
    }
    Tensor c = empty({M, N}, out_type, a);
    const Bias bias(bias_in, N);
    const int64_t need = scratch_for(M, N, K, block);
    const Tensor ws = need <= 0 ? Tensor() : scratch.defined() && (int64_t)scratch.nbytes() >= need ? scratch : empty({need}, at::kByte, a);
    int rc = gemm_raw((const int8_t *)a.data_ptr(), (const float *)sx.data_ptr(), ld_of(a), (const int8_t *)w.data_ptr(), (const float *)sw.data_ptr(), ld_of(w), bias,
                      c.data_ptr(), float_code(c), M, N, K, kw, block, need > 0 ? ws.data_ptr() : nullptr, need, stream_of(a));
    if (rc == BI8_ERR_UNSUPPORTED && kw != K) {
        // rows too far apart for the kernels' 32-bit offsets
        const int64_t extra = K / block - sw.size(0);
        w = at::constant_pad_nd(w, {0, K - w.size(1)});
        if (extra > 0) sw = at::constant_pad_nd(sw, {0, 0, 0, extra});
        rc = gemm_raw((const int8_t *)a.data_ptr(), (const float *)sx.data_ptr(), ld_of(a), (const int8_t *)w.data_ptr(), (const float *)sw.data_ptr(), ld_of(w), bias,
                      c.data_ptr(), float_code(c), M, N, K, K, block, need > 0 ? ws.data_ptr() : nullptr, need, stream_of(a));
    }
    check(rc, "bi8x_gemm");
    return c;
}

// ---- the layer ------------------------------------------------------------------------------------------------------
struct Config {
    int64_t block;
    ScalarType out_type, scale_type;
};

// Codes and scales side by side in one byte tensor: rows of `ld` codes, the scales behind them.
struct Packed {
    int64_t rows = 0, ld = 0, blocks = 0, at = 0;     // at = byte offset of the codes
    int64_t scales_at() const { return at + up(rows * ld, 256); }
    int64_t end() const { return up(scales_at() + blocks * rows * 4, 256); }
    int8_t *codes(const Tensor &t) const { return (int8_t *)t.data_ptr() + at; }
    float *scales(const Tensor &t) const { return (float *)((uint8_t *)t.data_ptr() + scales_at()); }
};
Packed pack(int64_t rows, int64_t contraction, int64_t block, int64_t at = 0) {
    const int64_t ld = up(contraction, 128);
    return Packed{rows, ld, ld / block, at};
}
// scales that are kept in another type are rounded to it once
void round_scales(const Tensor &t, const Packed &p, ScalarType type) {
    if (type == at::kFloat) return;
    Tensor s = t.slice(0, p.scales_at(), p.scales_at() + p.blocks * p.rows * 4).view(at::kFloat);
    s.copy_(s.to(type));
}
Bi8DualTask dual_task(const Tensor &x, const Tensor &qt_in, const Packed &q, const Tensor &t, const Packed &qt) {
    return Bi8DualTask{x.data_ptr(), q.codes(t), qt.codes(qt_in), q.scales(t), qt.scales(qt_in), x.size(0), x.size(1), ld_of(x), q.ld, qt.ld, qt.ld, q.ld};
}
void quantize_rows(const Tensor &x, const Tensor &t, const Packed &q, const Config &cfg, void *stream) {
    check(bi8x_quantize_rowwise(x.data_ptr(), float_code(x), q.codes(t), q.scales(t), x.size(0), x.size(1), q.ld, ld_of(x), q.ld, (int)cfg.block, stream),
          "bi8x_quantize_rowwise");
    round_scales(t, q, cfg.scale_type);
}

// Codes of a weight made ahead of the call, int8 [N,K] with contiguous rows, as a GEMM operand that only A is padded for.
bool ready_operand(const Tensor &w, int64_t contraction, int64_t block) {
    return fast_block(block) && (contraction % 128 == 0 || block != 32) && ld_of(w) % 16 == 0 && (uintptr_t)w.data_ptr() % 16 == 0 && whole_chunks(w, contraction);
}
// ... and the copy of one that is none, padded itself
std::pair<Tensor, Tensor> padded_operand(const Tensor &w, const Tensor &s, int64_t contraction, int64_t block) {
    const int64_t kp = up(contraction, 128), extra = kp / block - s.size(0);
    return {at::constant_pad_nd(w, {0, kp - contraction}).contiguous(), extra > 0 ? at::constant_pad_nd(s, {0, 0, 0, extra}) : s};
}
// y = a @ w.T on codes that are a packed operand and a ready one (or any, which is then copied)
void multiply_ready(const Packed &aq, const Tensor &t, const Tensor &w_in, const Tensor &state, int64_t contraction, const Bias &bias, const Tensor &out, int64_t M, int64_t N,
                    int64_t block, void *ws, int64_t need, void *stream) {
    const Tensor w = rows_of(w_in), s = scales_in(state);      // (scales kept in another type are converted, the codes are not touched)
    if (!pad_contraction(M, N, contraction, block) || (small_product(M, N, contraction) && (ld_of(w) % 16 != 0 || (uintptr_t)w.data_ptr() % 16 != 0)))
        return check(gemm_raw(aq.codes(t), aq.scales(t), aq.ld, (const int8_t *)w.data_ptr(), (const float *)s.data_ptr(), ld_of(w), bias, out.data_ptr(), float_code(out),
                              M, N, contraction, contraction, block, nullptr, 0, stream),
                     "bi8x_gemm");
    if (ready_operand(w, contraction, block)) {
        const int rc = gemm_raw(aq.codes(t), aq.scales(t), aq.ld, (const int8_t *)w.data_ptr(), (const float *)s.data_ptr(), ld_of(w), bias, out.data_ptr(), float_code(out), M,
                                N, aq.ld, up(contraction, 16), block, ws, need, stream);
        if (rc != BI8_ERR_UNSUPPORTED) return check(rc, "bi8x_gemm");    // (rows too far apart for the kernels' 32-bit offsets: copied)
    }
    const auto [wp, sp] = padded_operand(w, s, contraction, block);
    check(gemm_raw(aq.codes(t), aq.scales(t), aq.ld, (const int8_t *)wp.data_ptr(), (const float *)sp.data_ptr(), aq.ld, bias, out.data_ptr(), float_code(out), M, N, aq.ld, aq.ld,
                   block, ws, need, stream),
          "bi8x_gemm");
}
void check_codes(const Tensor &w, const Tensor &state, int64_t contraction, int64_t block) {
    require(w.is_cuda() && state.is_cuda(), "operands must be device tensors");
    require(w.scalar_type() == at::kChar && w.dim() == 2, "operands must be int8 codes");
    require(w.size(1) == contraction, "incompatible dimensions");
    require(state.dim() == 2 && state.size(0) == ceil_div(contraction, block) && state.size(1) == w.size(0), "scale shapes must be [ceil(K/block), rows]");
}

// What a forward pass keeps for the backward pass of X and of W: their codes along the other direction, [K,M] and [K,N].
struct Kept {
    Tensor codes, scales;              // packed: both in `codes`, W's behind X's in one tensor where both are kept
    bool packed = true;
};

// y = x @ W.T + bias.  `w` is the float weight, quantized here, or undefined where its codes come ready (w_int8, w_state).  Where the
// backward pass will want them, X and W are quantized along the other direction by the same read (need_xt, need_wt).
Tensor linear_forward(const Tensor &x_in, const Tensor &w_in, const Tensor &w_int8, const Tensor &w_state, const Tensor &bias_in, const Config &cfg, bool need_xt, bool need_wt,
                      Kept &xt, Kept &wt) {
    const Tensor x = matrix_of(x_in), w = w_in.defined() ? rows_of(w_in) : w_in;
    const int x_code = float_code(x), w_code = w.defined() ? float_code(w) : 0;
    const int64_t M = x.size(0), K = x.size(1), N = w.defined() ? w.size(0) : w_int8.size(0), B = cfg.block;
    if (w.defined()) require(w.is_cuda() && w.dim() == 2 && w.size(1) == K, "incompatible dimensions");
    else check_codes(w_int8, w_state, K, B);
    void *const stream = stream_of(x);

    if (fast_block(B) && M > 0 && N > 0 && K > 0) {
        Tensor out = empty(with_last(x_in, N), cfg.out_type, x);
        const Bias bias(bias_in, N);
        // a few rows against codes that are ready: one launch, where the library covers it
        if (M >= 3 && M <= 16 && !w.defined() && !need_xt && x_code == dtype_code(cfg.out_type) && cfg.scale_type == at::kFloat && w_state.scalar_type() == at::kFloat &&
            w_state.is_contiguous() && w_int8.stride(1) == 1) {
            const int rc = bi8x_linear_rows(x.data_ptr(), x_code, (const int8_t *)w_int8.data_ptr(), (const float *)w_state.data_ptr(), bias.ptr, bias.code, out.data_ptr(), M,
                                            N, K, ld_of(x), ld_of(w_int8), N, (int)B, stream);
            if (rc == BI8_OK) return out;
            if (rc != BI8_ERR_UNSUPPORTED) check(rc, "bi8x_linear_rows");
        }
        // one allocation for what does not outlive the call
        const Packed xq = pack(M, K, B), wq = pack(w.defined() ? N : 0, K, B, xq.end()), xtq = pack(K, M, B), wtq = pack(K, N, B, need_xt ? xtq.end() : 0);
        const bool pad = pad_contraction(M, N, K, B);
        const int64_t kp = pad ? xq.ld : K, need = pad ? scratch_for(M, N, kp, B) : 0, ws_at = wq.end();
        const Tensor t = empty({ws_at + need}, at::kByte, x);
        // ... and one for what is kept
        if (need_xt) xt.codes = empty({need_wt ? wtq.end() : xtq.end()}, at::kByte, x);
        if (need_wt) wt.codes = need_xt ? xt.codes : empty({wtq.end()}, at::kByte, x);
        Bi8DualTask task[2];
        int n = 0;
        if (need_xt) task[n++] = dual_task(x, xt.codes, xq, t, xtq);
        if (need_wt) task[n++] = dual_task(w, wt.codes, wq, t, wtq);
        if (n == 2 && x_code != w_code) {
            check(bi8x_quantize_dual(task + 1, 1, w_code, (int)B, nullptr, stream), "bi8x_quantize_dual");
            n = 1;
        }
        if (n > 0) check(bi8x_quantize_dual(task, n, need_xt ? x_code : w_code, (int)B, nullptr, stream), "bi8x_quantize_dual");
        if (need_xt) {
            round_scales(t, xq, cfg.scale_type);
            round_scales(xt.codes, xtq, cfg.scale_type);
        } else {
            quantize_rows(x, t, xq, cfg, stream);
        }
        if (need_wt) {
            round_scales(t, wq, cfg.scale_type);
            round_scales(wt.codes, wtq, cfg.scale_type);
        } else if (w.defined()) {
            quantize_rows(w, t, wq, cfg, stream);
        }
        void *const ws = need > 0 ? (uint8_t *)t.data_ptr() + ws_at : nullptr;
        if (w.defined()) {
            check(gemm_raw(xq.codes(t), xq.scales(t), xq.ld, wq.codes(t), wq.scales(t), wq.ld, bias, out.data_ptr(), float_code(out), M, N, kp, kp, B, ws, need, stream), "bi8x_gemm");
        } else {
            multiply_ready(xq, t, w_int8, w_state, K, bias, out, M, N, B, ws, need, stream);
        }
        return out;
    }

    // other block sizes, empty operands: the single-direction quantizers and the GEMM that copies what it has to
    auto [xq, xs] = quantize_rowwise(x, B, cfg.scale_type);
    if (need_xt) {
        std::tie(xt.codes, xt.scales) = quantize_transposed(x, B, cfg.scale_type);
        xt.packed = false;
    }
    Tensor wq = w_int8, ws = w_state;
    if (w.defined()) std::tie(wq, ws) = quantize_rowwise(w, B, cfg.scale_type);
    if (need_wt) {
        std::tie(wt.codes, wt.scales) = quantize_transposed(w, B, cfg.scale_type);
        wt.packed = false;
    }
    return gemm(xq, rows_of(wq), xs, ws, bias_in, B, cfg.out_type).view(with_last(x_in, N));
}

// What a backward pass needs to know besides the codes: autograd's node keeps it.
struct Shape {
    Config cfg;
    int64_t M = 0, K = 0, N = 0;
    std::vector<int64_t> x_sizes;
    bool wt_packed = true, together = false;       // together: W's codes are behind X's in one tensor
};

// grad_X [M,K] = G [M,N] @ W [N,K], contracted over N; grad_W [N,K] = G.T [N,M] @ X [M,K], contracted over the rows
// (block_linear.py:88-112); grad_bias = the column sums of G.  held: codes and scales of X transposed, of W transposed.
torch::autograd::variable_list linear_backward(const Tensor &G_in, const Shape &s, const Tensor *held, bool need_gx, bool need_gw, bool need_gb) {
    torch::autograd::variable_list result(3);
    const Config &cfg = s.cfg;
    const int64_t M = s.M, K = s.K, N = s.N;
    const bool graph = at::GradMode::is_enabled();
    at::AutoGradMode no_grad(false);
    require(G_in.is_cuda(), "the gradient must be a device tensor");
    c10::DeviceGuard guard(G_in.device());
    const Tensor G = matrix_of(G_in);
    const int g_code = float_code(G);
    const int64_t B = cfg.block;
    void *const stream = stream_of(G);
    const Packed xtq = pack(K, M, B), wtq = pack(K, N, B, s.together ? xtq.end() : 0);

    if (fast_block(B) && M > 0 && N > 0 && K > 0 && (need_gx || need_gw)) {
        const Packed gq = pack(need_gx ? M : 0, N, B), gtq = pack(need_gw ? N : 0, M, B, gq.end());
        const bool both = need_gx && need_gw, sums = both && need_gb;
        const int64_t part_at = gtq.end(), ws_at = up(part_at + (sums ? bi8_colsum_workspace_bytes(M, N) : 0), 256);
        const int64_t kx = pad_contraction(M, K, N, B) ? gq.ld : N, kw = pad_contraction(N, K, M, B) ? gtq.ld : M;      // the contractions as multiplied
        const int64_t need1 = need_gx && kx == gq.ld ? scratch_for(M, K, kx, B) : 0, need2 = need_gw && kw == gtq.ld ? scratch_for(N, K, kw, B) : 0;
        const Tensor t = empty({ws_at + std::max(need1, need2)}, at::kByte, G);
        uint8_t *const base = (uint8_t *)t.data_ptr();
        if (both) {
            const Bi8DualTask task = dual_task(G, t, gq, t, gtq);
            check(bi8x_quantize_dual(&task, 1, g_code, (int)B, sums ? (float *)(base + part_at) : nullptr, stream), "bi8x_quantize_dual");
            round_scales(t, gq, cfg.scale_type);
            round_scales(t, gtq, cfg.scale_type);
        } else if (need_gx) {
            quantize_rows(G, t, gq, cfg, stream);
        } else {
            if (gtq.ld != M) t.slice(0, 0, gtq.end()).zero_();       // (the single-direction quantizer writes no padding)
            check(bi8_quantize_transposed(G.data_ptr(), g_code, gtq.codes(t), gtq.scales(t), M, N, ld_of(G), gtq.ld, (int)B, stream), "bi8_quantize_transposed");
            round_scales(t, gtq, cfg.scale_type);
        }
        const Bias none(Tensor(), 0);
        Tensor gx = need_gx ? empty(s.x_sizes, cfg.out_type, G) : Tensor(), gw = need_gw ? empty({N, K}, cfg.out_type, G) : Tensor();
        if (sums) result[2] = empty({N}, G.scalar_type(), G);
        const Bi8ColSums col_sums{(const float *)(base + part_at), sums ? result[2].data_ptr() : nullptr, g_code, M, N};
        bool paired = false;                       // both in one launch, where the library would have it so
        if (both && kx == gq.ld && kw == gtq.ld) {
            const Tensor w = s.wt_packed ? Tensor() : rows_of(held[2]), ws = s.wt_packed ? Tensor() : scales_in(held[3]);
            if (s.wt_packed || ready_operand(w, N, B)) {
                const Bi8Gemm pair[2] = {{gq.codes(t), s.wt_packed ? wtq.codes(held[2]) : (const int8_t *)w.data_ptr(), gq.scales(t),
                                          s.wt_packed ? wtq.scales(held[2]) : (const float *)ws.data_ptr(), gx.data_ptr(), M, K, kx, s.wt_packed ? kx : up(N, 16), gq.ld,
                                          s.wt_packed ? wtq.ld : ld_of(w), std::max<int64_t>(K, 1)},
                                         {gtq.codes(t), xtq.codes(held[0]), gtq.scales(t), xtq.scales(held[0]), gw.data_ptr(), N, K, kw, kw, gtq.ld, xtq.ld, std::max<int64_t>(K, 1)}};
                const int rc = bi8x_gemm_pair(pair, float_code(gx), (int)B, sums ? &col_sums : nullptr, stream);
                if (rc != BI8_ERR_UNSUPPORTED) check(rc, "bi8x_gemm_pair");
                paired = rc == BI8_OK;
            }
        }
        if (need_gx && !paired) {
            void *const ws = need1 > 0 ? base + ws_at : nullptr;
            if (s.wt_packed) {
                check(gemm_raw(gq.codes(t), gq.scales(t), gq.ld, wtq.codes(held[2]), wtq.scales(held[2]), wtq.ld, none, gx.data_ptr(), float_code(gx), M, K, kx, kx, B,
                               ws, need1, stream),
                      "bi8x_gemm");
            } else {
                multiply_ready(gq, t, held[2], held[3], N, none, gx, M, K, B, ws, need1, stream);
            }
        }
        if (need_gw && !paired) {
            const Bi8Gemm q{gtq.codes(t), xtq.codes(held[0]), gtq.scales(t), xtq.scales(held[0]), gw.data_ptr(), N, K, kw, kw, gtq.ld, xtq.ld, std::max<int64_t>(K, 1)};
            void *const ws = need2 > 0 ? base + ws_at : nullptr;
            if (sums) check(bi8x_gemm_sums(&q, float_code(gw), (int)B, ws, need2, &col_sums, stream), "bi8x_gemm_sums");
            else check(gemm_raw(q.A, q.sA, q.lda, q.W, q.sW, q.ldw, none, q.C, float_code(gw), N, K, kw, kw, B, ws, need2, stream), "bi8x_gemm");
        }
        result[0] = gx;
        result[1] = gw;
    } else {
        if (need_gx) {
            auto [q, qs] = quantize_rowwise(G, B, cfg.scale_type);
            result[0] = gemm(q, rows_of(held[2]), qs, held[3], Tensor(), B, cfg.out_type).view(s.x_sizes);
        }
        if (need_gw) {
            auto [q, qs] = quantize_transposed(G, B, cfg.scale_type);
            result[1] = gemm(q, held[0], qs, held[1], Tensor(), B, cfg.out_type);
        }
    }
    if (need_gb && !result[2].defined()) {
        at::AutoGradMode as_called(graph);         // (plain torch operators: differentiable under create_graph)
        result[2] = G_in.reshape({M, N}).sum(0);
    }
    return result;
}

// The same node for compiled autograd, which asks a node to describe itself and to run on stand-ins: torch's C++ autograd functions can.
// (Not used in eager mode: an autograd function of torch costs the host 1.4 us more in the forward pass and 1.1 us in the backward.)
struct CompiledBackward : public torch::autograd::Function<CompiledBackward> {
    static torch::autograd::variable_list backward(torch::autograd::AutogradContext *ctx, torch::autograd::variable_list grads) {
        torch::autograd::variable_list held = ctx->get_saved_variables();
        const std::vector<int64_t> of = ctx->saved_data["of"].toIntVector();
        const Shape s{{of[0], (ScalarType)of[1], (ScalarType)of[2]}, of[3], of[4], of[5], {of.begin() + 9, of.end()}, of[6] != 0, of[7] != 0};
        if (s.together) held[2] = held[0];
        if (!grads[0].defined()) {
            std::vector<int64_t> size = s.x_sizes;
            size.back() = s.N;
            grads[0] = at::zeros(size, at::TensorOptions().dtype(s.cfg.out_type).device(at::kCUDA, (c10::DeviceIndex)of[8]));
        }
        return linear_backward(grads[0], s, held.data(), held[2].defined() && ctx->needs_input_grad(0), held[0].defined() && ctx->needs_input_grad(1), ctx->needs_input_grad(2));
    }
};

struct LinearBackward : public torch::autograd::Node {
    using Compiled = torch::autograd::CppNode<CompiledBackward>;
    Shape s;
    c10::DeviceIndex device = 0;
    torch::autograd::SavedVariable saved[4];
    bool has[4] = {false, false, false, false}, freed = false;
    mutable std::shared_ptr<Compiled> compiled;

    std::string name() const override { return "BlockInt8LinearBackward"; }
    void keep(const Kept &xt, const Kept &wt) {
        s.wt_packed = wt.packed;
        s.together = wt.packed && xt.codes.defined() && wt.codes.is_same(xt.codes);
        const Tensor *t[4] = {&xt.codes, &xt.scales, &wt.codes, &wt.scales};
        for (int i = 0; i < 4; ++i) {
            has[i] = t[i]->defined() && !(i == 2 && s.together);
            if (has[i]) saved[i] = torch::autograd::SavedVariable(*t[i], false);
        }
    }
    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        freed = true;
        compiled.reset();
        for (auto &v : saved) v.reset_data();
    }
    void unpack(Tensor *held, const std::shared_ptr<torch::autograd::Node> &self) const {
        TORCH_CHECK(!freed, torch::autograd::ERR_BACKWARD_TWICE);
        for (int i = 0; i < 4; ++i)
            if (has[i]) held[i] = saved[i].unpack(self);
    }
    torch::autograd::variable_list apply(torch::autograd::variable_list &&grads) override {
        // (no gradient reached the output: zeros, as an autograd function of torch gets them)
        if (!grads[0].defined()) grads[0] = input_metadata(0).zeros_like();
        Tensor held[4];
        {
            std::lock_guard<std::mutex> lock(mutex_);
            unpack(held, shared_from_this());
        }
        if (s.together) held[2] = held[0];
        return linear_backward(grads[0], s, held, held[2].defined() && task_should_compute_output(0), held[0].defined() && task_should_compute_output(1),
                               task_should_compute_output(2));
    }
    void compiled_args(torch::dynamo::autograd::CompiledNodeArgs &args) const override {
        torch::autograd::variable_list held(4);
        unpack(held.data(), std::const_pointer_cast<torch::autograd::Node>(shared_from_this()));
        compiled = std::shared_ptr<Compiled>(new Compiled(), torch::autograd::deleteNode);
        compiled->set_ctx_grad_fn(compiled);
        compiled->set_next_edges(torch::autograd::edge_list(next_edges()));
        compiled->is_variable_input_ = {true, true, true};
        std::vector<int64_t> of = {s.cfg.block, (int64_t)s.cfg.out_type, (int64_t)s.cfg.scale_type, s.M, s.K, s.N, s.wt_packed, s.together, device};
        of.insert(of.end(), s.x_sizes.begin(), s.x_sizes.end());
        compiled->ctx_.saved_data["of"] = std::move(of);
        compiled->ctx_.set_materialize_grads(false);
        compiled->ctx_.save_for_backward(std::move(held));
        compiled->save_variables_to_ctx();
        compiled->compiled_args(args);
    }
    torch::autograd::variable_list apply_with_saved(const torch::autograd::variable_list &grads, torch::dynamo::autograd::SwapSavedVariables &swapped) override {
        return compiled->apply_with_saved(grads, swapped);
    }
};

// The differentiable layer: autograd's inputs are x, `stands_for_w` (the tensor that receives grad_W: the float weight itself, or what
// stands for it where its codes come ready) and the bias.
Tensor linear_apply(const Tensor &x, const Tensor &w, const Tensor &w_int8, const Tensor &w_state, const Tensor &stands_for_w, const Kept &wt_ready, const Tensor &bias,
                    const Config &cfg) {
    require(x.is_cuda(), "x must be a device tensor");
    for (const Tensor *t : {&x, &w, &stands_for_w, &bias})
        TORCH_CHECK_NOT_IMPLEMENTED(!t->defined() || !t->_fw_grad(0).defined(), "blockwise_int8_linear has no forward-mode derivative");
    const bool grad = at::GradMode::is_enabled();
    const bool need_gx = grad && x.requires_grad(), need_gw = grad && stands_for_w.defined() && stands_for_w.requires_grad(), need_gb = grad && bias.defined() && bias.requires_grad();
    c10::DeviceGuard guard(x.device());
    Kept xt, wt;
    Tensor out;
    {
        at::AutoGradMode no_grad(false);
        out = linear_forward(x, w, w_int8, w_state, bias, cfg, need_gw, need_gx && w.defined(), xt, wt);
    }
    if (need_gx || need_gw || need_gb) {
        std::shared_ptr<LinearBackward> node(new LinearBackward(), torch::autograd::deleteNode);
        node->set_next_edges(torch::autograd::collect_next_edges(x, stands_for_w, bias));
        node->s.cfg = cfg;
        node->s.K = x.size(-1);
        node->s.N = out.size(-1);
        node->s.M = 1;
        for (int64_t d = 0; d + 1 < x.dim(); ++d) node->s.M *= x.size(d);
        node->s.x_sizes.assign(x.sizes().begin(), x.sizes().end());
        node->device = x.device().index();
        node->keep(xt, w.defined() || !need_gx ? wt : wt_ready);
        torch::autograd::set_history(out, node);
    }
    return out;
}

// Quantize + GEMM in one launch for one or two rows, where the library covers it (bi8_linear_few_rows); undefined otherwise.
Tensor few_rows(const Tensor &x_in, const Tensor &w, const Tensor &state, const Tensor &bias_in, int64_t block, ScalarType out_type) {
    if (x_in.scalar_type() != out_type || dtype_code(out_type) < 0 || w.scalar_type() != at::kChar || state.scalar_type() != at::kFloat || !state.is_contiguous() ||
        w.dim() != 2 || w.stride(1) != 1 || x_in.size(-1) != w.size(1) || state.dim() != 2 || state.size(1) != w.size(0) || state.size(0) != ceil_div(w.size(1), block))
        return Tensor();
    require(x_in.is_cuda() && w.is_cuda() && state.is_cuda(), "operands must be device tensors");
    const Tensor x = matrix_of(x_in);              // (also rows that overlap, an expanded row for instance, become rows)
    const int64_t M = x.size(0), K = x.size(1), N = w.size(0);
    if (M < 1 || M > 2 || (block != 64 && block != 128) || K % 128 != 0 || N < 1 || K < 1) return Tensor();
    c10::DeviceGuard guard(x.device());
    const Bias bias(bias_in, N);
    Tensor out = empty(with_last(x_in, N), out_type, x);
    const int rc = bi8_linear_few_rows(x.data_ptr(), dtype_code(out_type), (const int8_t *)w.data_ptr(), (const float *)state.data_ptr(), bias.ptr, bias.code, out.data_ptr(), M,
                                       N, K, ld_of(x), ld_of(w), N, (int)block, stream_of(x));
    if (rc == BI8_ERR_UNSUPPORTED) return Tensor();        // alignment of a view, for instance
    check(rc, "bi8_linear_few_rows");
    return out;
}

// ---- Python ---------------------------------------------------------------------------------------------------------
PyObject *bi8_error = nullptr;

struct Args {
    PyObject *const *v;
    Py_ssize_t n;
    const char *what;
    Tensor tensor(int i) const {
        if (!THPVariable_Check(v[i])) throw TypeFailure(std::string(what) + ": argument " + std::to_string(i + 1) + " must be a tensor");
        return THPVariable_Unpack(v[i]);
    }
    Tensor optional_tensor(int i) const { return v[i] == Py_None ? Tensor() : tensor(i); }
    int64_t integer(int i) const {
        const int64_t r = PyLong_AsLongLong(v[i]);
        if (r == -1 && PyErr_Occurred()) {
            PyErr_Clear();
            throw TypeFailure(std::string(what) + ": argument " + std::to_string(i + 1) + " must be an integer");
        }
        return r;
    }
    int64_t block(int i) const {
        const int64_t b = integer(i);
        if (b < 1 || b > (1 << 20)) check(BI8_ERR_BAD_BLOCK, what);
        return b;
    }
    ScalarType dtype(int i) const {
        if (!THPDtype_Check(v[i])) throw TypeFailure(std::string(what) + ": argument " + std::to_string(i + 1) + " must be a dtype");
        return ((THPDtype *)v[i])->scalar_type;
    }
};

// Runs f without the interpreter lock; its failures become Python exceptions.
template <class F> auto without_gil(F &&f) {
    struct Release {
        PyThreadState *state = PyEval_SaveThread();
        ~Release() { PyEval_RestoreThread(state); }
    } release;
    return f();
}
PyObject *wrapped(const Tensor &t) {
    if (!t.defined()) Py_RETURN_NONE;
    return THPVariable_Wrap(t);
}
PyObject *wrapped(const std::pair<Tensor, Tensor> &p) {
    PyObject *t = PyTuple_New(2);
    if (t) {
        PyTuple_SET_ITEM(t, 0, THPVariable_Wrap(p.first));
        PyTuple_SET_ITEM(t, 1, THPVariable_Wrap(p.second));
    }
    return t;
}
template <class F> PyObject *guarded(const char *what, Py_ssize_t want, PyObject *const *v, Py_ssize_t n, F &&f) {
    try {
        if (n != want) throw TypeFailure(std::string(what) + " takes " + std::to_string(want) + " arguments");
        return f(Args{v, n, what});
    } catch (python_error &e) {                        // raised by a saved-tensor hook (a checkpoint ends its recomputation so)
        e.restore();
    } catch (const Bi8Failure &e) {
        PyErr_SetString(bi8_error ? bi8_error : PyExc_RuntimeError, e.what());
    } catch (const OperandError &e) {
        PyErr_SetString(PyExc_AssertionError, e.what());
    } catch (const TypeFailure &e) {
        PyErr_SetString(PyExc_TypeError, e.what());
    } catch (const c10::OutOfMemoryError &e) {
        PyObject *cls = nullptr, *mod = PyImport_ImportModule("torch");
        if (mod) cls = PyObject_GetAttrString(mod, "OutOfMemoryError");
        PyErr_SetString(cls ? cls : PyExc_RuntimeError, e.what_without_backtrace());
        Py_XDECREF(cls);
        Py_XDECREF(mod);
    } catch (const c10::NotImplementedError &e) {
        PyErr_SetString(PyExc_NotImplementedError, e.what_without_backtrace());
    } catch (const c10::Error &e) {
        PyErr_SetString(PyExc_RuntimeError, e.what_without_backtrace());
    } catch (const std::exception &e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
    }
    return nullptr;
}

PyObject *py_quantize_rowwise(PyObject *, PyObject *const *v, Py_ssize_t n) {       // x, block, scale dtype
    return guarded("quantize_rowwise", 3, v, n, [](Args a) {
        const Tensor x = a.tensor(0);
        const int64_t block = a.block(1);
        const ScalarType st = a.dtype(2);
        return wrapped(without_gil([&] {
            at::AutoGradMode no_grad(false);
            return quantize_rowwise(x, block, st);
        }));
    });
}
PyObject *py_quantize_transposed(PyObject *, PyObject *const *v, Py_ssize_t n) {    // x, block, scale dtype
    return guarded("quantize_transposed", 3, v, n, [](Args a) {
        const Tensor x = a.tensor(0);
        const int64_t block = a.block(1);
        const ScalarType st = a.dtype(2);
        return wrapped(without_gil([&] {
            at::AutoGradMode no_grad(false);
            return quantize_transposed(x, block, st);
        }));
    });
}
PyObject *py_dequantize(PyObject *, PyObject *const *v, Py_ssize_t n) {             // codes, scales, block, output dtype
    return guarded("dequantize", 4, v, n, [](Args a) {
        const Tensor q = a.tensor(0), s = a.tensor(1);
        const int64_t block = a.block(2);
        const ScalarType ot = a.dtype(3);
        return wrapped(without_gil([&] {
            at::AutoGradMode no_grad(false);
            return dequantize(q, s, block, ot);
        }));
    });
}
PyObject *py_gemm(PyObject *, PyObject *const *v, Py_ssize_t n) {                   // a [M,K], b [K,N], scales of both, bias, block, output dtype, scratch
    return guarded("gemm", 8, v, n, [](Args a) {
        const Tensor A = a.tensor(0), b = a.tensor(1), sx = a.tensor(2), sw = a.tensor(3), bias = a.optional_tensor(4), scratch = a.optional_tensor(7);
        const int64_t block = a.block(5);
        const ScalarType ot = a.dtype(6);
        return wrapped(without_gil([&] {
            at::AutoGradMode no_grad(false);
            return gemm(rows_of(A), rows_of(b.t()), sx, sw, bias, block, ot, scratch);
        }));
    });
}
PyObject *py_linear(PyObject *, PyObject *const *v, Py_ssize_t n) {                 // x, weight, bias, block, output dtype, scale dtype
    return guarded("linear", 6, v, n, [](Args a) {
        const Tensor x = a.tensor(0), w = a.tensor(1), bias = a.optional_tensor(2);
        const Config cfg{a.block(3), a.dtype(4), a.dtype(5)};
        return wrapped(without_gil([&] { return linear_apply(x, w, Tensor(), Tensor(), w, Kept(), bias, cfg); }));
    });
}
// x, W codes, W scales, bias, transposed W codes, their scales, weight or None, block, output dtype, scale dtype
PyObject *py_linear_kept(PyObject *, PyObject *const *v, Py_ssize_t n) {
    return guarded("linear_kept", 10, v, n, [](Args a) {
        const Tensor x = a.tensor(0), wq = a.tensor(1), ws = a.tensor(2), bias = a.optional_tensor(3), weight = a.optional_tensor(6);
        Kept wt;
        wt.codes = a.tensor(4);
        wt.scales = a.tensor(5);
        wt.packed = false;
        const Config cfg{a.block(7), a.dtype(8), a.dtype(9)};
        return wrapped(without_gil([&] {
            check_codes(wt.codes, wt.scales, wq.size(0), cfg.block);
            return linear_apply(x, Tensor(), wq, ws, weight, wt, bias, cfg);
        }));
    });
}
PyObject *py_infer(PyObject *, PyObject *const *v, Py_ssize_t n) {                  // x, W codes, W scales, bias, block, output dtype, scale dtype
    return guarded("infer", 7, v, n, [](Args a) {
        const Tensor x = a.tensor(0), wq = a.tensor(1), ws = a.tensor(2), bias = a.optional_tensor(3);
        const Config cfg{a.block(4), a.dtype(5), a.dtype(6)};
        return wrapped(without_gil([&] {
            at::AutoGradMode no_grad(false);
            require(x.is_cuda(), "x must be a device tensor");
            c10::DeviceGuard guard(x.device());
            Kept xt, wt;
            return linear_forward(x, Tensor(), wq, ws, bias, cfg, false, false, xt, wt);
        }));
    });
}
PyObject *py_few_rows(PyObject *, PyObject *const *v, Py_ssize_t n) {               // x, W codes, W scales, bias, block, dtype -> output or None
    return guarded("few_rows", 6, v, n, [](Args a) {
        const Tensor x = a.tensor(0), wq = a.tensor(1), ws = a.tensor(2), bias = a.optional_tensor(3);
        const int64_t block = a.block(4);
        const ScalarType ot = a.dtype(5);
        return wrapped(without_gil([&] {
            at::AutoGradMode no_grad(false);
            return few_rows(x, wq, ws, bias, block, ot);
        }));
    });
}
PyObject *py_set_error(PyObject *, PyObject *cls) {
    Py_INCREF(cls);
    Py_XDECREF(bi8_error);
    bi8_error = cls;
    Py_RETURN_NONE;
}

#define BI8_METHOD(name) {#name, (PyCFunction)(void (*)(void))py_##name, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {BI8_METHOD(quantize_rowwise), BI8_METHOD(quantize_transposed), BI8_METHOD(dequantize), BI8_METHOD(gemm), BI8_METHOD(linear),
                         BI8_METHOD(linear_kept), BI8_METHOD(infer), BI8_METHOD(few_rows), {"set_error", py_set_error, METH_O, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_bi8_torch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__bi8_torch(void) { return PyModule_Create(&module); }

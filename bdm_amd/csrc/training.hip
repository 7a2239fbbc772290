// Backward of the layer's elementwise work around its projection GEMMs under
// autograd: the controllers (heads.py:11-22, _parameters.py:189-220), the
// output interface before o_proj (_parameters.py:222-232) and the product-key
// softmax (gdn2_banks.py:104-114).  Each is the derivative of the values that
// the forward kernels (epilogue.hip, router.hip) store, formed in FP32 from the
// projections and rounded once, in one pass instead of the chains of
// elementwise, cast, reduce and scatter kernels that autograd makes of them.
// At 8,192 tokens, 1,024 columns, H8 S8 v128 the layer's training step (the
// input projected by the concatenated weights, apart from the output gate) took
// 2,370 us and takes 1,560: 46 us here for the controllers, 31 for the output
// interface and 6 for each role's routes, where the chains took ~600 us and the
// separate products' gradients ~600.
#include "epilogue_ops.h"

namespace bdm {
namespace {

// ------------------------------------------------------------ controllers

template <typename T>
struct ControllerGradParams {
    const T *proj, *f;
    const void *a_log, *dt_bias;
    const T *dq, *dk, *dv, *db, *dw, *dread, *dwrite, *dgate;
    const float *dg;
    T *dproj, *df;
    float *terms;
    int64_t proj_stride, f_stride;
    int q_col, k_col, v_col, b_col, w_col, read_col, write_col, gate_col;
    int heads, hv, route_width, param_dtype, qk_norm;
};

template <typename T>
__device__ __forceinline__ void sigmoid8(const float (&t)[8], float (&s)[8]) {
#pragma unroll
    for (int j = 0; j < 8; ++j) s[j] = sigmoid_f(t[j]);
}

// One workgroup per token; a thread takes items of 8 columns (S for the rows
// of a head): 4H rows of q, k, b, g, then the chunks of v, w, gate, read and
// write.  Bound: HBM, the projection and every gradient read once and the
// projection's gradient written once (40 MB of each at 8,192 tokens and the 2,432
// columns of H8 S8 v128, 256 banks, without the gate); the last three kinds are
// copies into the one gradient that the two backward GEMMs read.
template <typename T, int S>
__global__ __launch_bounds__(256) void controller_backward_kernel(ControllerGradParams<T> p) {
    const int64_t token = blockIdx.x;
    const T *row = p.proj + token * p.proj_stride;
    T *drow = p.dproj + token * p.proj_stride;
    const int total = p.heads * p.hv, vc = total / 8, rc = p.route_width / 8;
    const int wide = (p.dgate ? 3 : 2) * vc;  // v, w and, where the projection has it, the gate
    const int items = 4 * p.heads + wide + 2 * rc;
    const int64_t hs = int64_t(p.heads) * S;
    for (int it = threadIdx.x; it < items; it += int(blockDim.x)) {
        if (it < 4 * p.heads) {
            const int h = it % p.heads, kind = it / p.heads;
            if (kind == 3) {
                // g = -exp(A_log) softplus(z), z = f + dt_bias: dz = -dg exp(A_log) sigmoid(z), dA_log = sum dg g
                const float a = -expf(param_at(p.a_log, p.param_dtype, h));
#pragma unroll
                for (int r0 = 0; r0 < S; r0 += 8) {
                    float f[8], bias[8], dg[8], dz[8], rate[8];
                    load8<T, true>(p.f + token * p.f_stride + h * S + r0, f);
                    param8<true>(p.dt_bias, p.param_dtype, int64_t(h) * S + r0, bias);
                    load8<float, true>(p.dg + token * hs + h * S + r0, dg);
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        const float z = f[j] + bias[j];
                        dz[j] = dg[j] * a * (z > 20.f ? 1.f : 1.f / (1.f + expf(-z)));
                        rate[j] = dg[j] * (a * softplus_f(z));
                    }
                    store_row<8>(p.df + token * hs + h * S + r0, dz);
                    store_row<8>(p.terms + token * 2 * hs + h * S + r0, dz);
                    store_row<8>(p.terms + token * 2 * hs + hs + h * S + r0, rate);
                }
                continue;
            }
            const T *src = row + (kind == 0 ? p.q_col : (kind == 1 ? p.k_col : p.b_col)) + h * S;
            T *dst = drow + (src - row);
            const T *dy = (kind == 0 ? p.dq : (kind == 1 ? p.dk : p.db)) + token * hs + h * S;
            float d[S], t[S], s[S];
#pragma unroll
            for (int r0 = 0; r0 < S; r0 += 8) {
                float d8[8], t8[8], s8[8];
                load8<T, true>(src + r0, t8);
                load8<T, true>(dy + r0, d8);
                sigmoid8<T>(t8, s8);
#pragma unroll
                for (int j = 0; j < 8; ++j) d[r0 + j] = d8[j], t[r0 + j] = t8[j], s[r0 + j] = s8[j];
            }
            if (kind < 2) {
                // y = x inv of x = round(silu(t)): dx = inv (dy - y (y . dy)), the norm's guard as in qk_row
                float ss = 0.f, dot = 0.f, x[S];
#pragma unroll
                for (int r = 0; r < S; ++r) {
                    x[r] = round_to<T>(t[r] * s[r]);
                    ss = fmaf(x[r], x[r], ss);
                    dot = fmaf(x[r], d[r], dot);
                }
                const float norm = sqrtf(ss);
                const float inv = p.qk_norm == 1 ? rsqrtf(ss + 1e-6f) : 1.f / fmaxf(norm, 1e-12f);
                const float back = p.qk_norm == 1 || norm > 1e-12f ? dot * inv * inv : 0.f;
#pragma unroll
                for (int r = 0; r < S; ++r) d[r] = inv * (d[r] - x[r] * back) * s[r] * (1.f + t[r] * (1.f - s[r]));
            } else {
#pragma unroll
                for (int r = 0; r < S; ++r) d[r] *= s[r] * (1.f - s[r]);
            }
#pragma unroll
            for (int r0 = 0; r0 < S; r0 += 8) {
                float d8[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) d8[j] = d[r0 + j];
                store_row<8>(dst + r0, d8);
            }
            continue;
        }
        const int c = it - 4 * p.heads;
        const int kind = c < wide ? c / vc : 3 + (c - wide) / rc;  // v, w, gate, read, write
        const int col = (c < wide ? c % vc : (c - wide) % rc) * 8;
        if (kind >= 2) {
            const T *src = kind == 2 ? p.dgate + token * total : (kind == 3 ? p.dread : p.dwrite) + token * p.route_width;
            T *dst = drow + (kind == 2 ? p.gate_col : (kind == 3 ? p.read_col : p.write_col));
            float d[8];
            load8<T, true>(src + col, d);
            store_row<8>(dst + col, d);
            continue;
        }
        float t[8], d[8], s[8];
        const int at = (kind == 0 ? p.v_col : p.w_col) + col;
        load8<T, true>(row + at, t);
        load8<T, true>((kind == 0 ? p.dv : p.dw) + token * total + col, d);
        sigmoid8<T>(t, s);
#pragma unroll
        for (int j = 0; j < 8; ++j) d[j] *= kind == 0 ? s[j] * (1.f + t[j] * (1.f - s[j])) : s[j] * (1.f - s[j]);
        store_row<8>(drow + at, d);
    }
}

// --------------------------------------------------------- output interface

template <typename T>
struct OutputGradParams {
    const T *raw, *gate, *dy;
    const void *weight, *bias;
    T *draw, *dgate;
    float *partials;  // [blocks, 2 * width]: d weight, d bias
    int64_t tokens, gate_stride;
    int width, param_dtype, norm_kind;
    float eps;
};

constexpr int kOutputRows = 32;  // tokens of a workgroup

// out = round(n) * round(sigmoid(gate)), n the layer or RMS normalization of
// raw.  One wave per token, a lane owns 8-column chunks as in
// output_epilogue_kernel; the waves of a workgroup take kOutputRows tokens and
// keep the parameters' gradients in registers, added over the waves in LDS and
// over the workgroups by column_sum_kernel.  Bound: HBM, three rows read and
// two written per token.
template <typename T, int MAXC>
__global__ __launch_bounds__(256) void output_backward_kernel(OutputGradParams<T> p) {
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave, waves = blockDim.x / kWave;
    const int64_t first = int64_t(blockIdx.x) * kOutputRows, last = min(p.tokens, first + kOutputRows);
    const float inv_n = 1.f / float(p.width);
    const bool layer = p.norm_kind == 1;
    float dweight[MAXC][8] = {}, dbias[MAXC][8] = {};
    for (int64_t token = first + wave; token < last; token += waves) {
        float x[MAXC][8], gs[MAXC][8], d[MAXC][8];
        float sum = 0.f, sq = 0.f;
#pragma unroll
        for (int i = 0; i < MAXC; ++i) {
            const int c = min((lane + i * kWave) * 8, p.width - 8);  // chunks past the width re-read the last
            const bool live = (lane + i * kWave) * 8 < p.width;
            load8<T, true>(p.raw + token * p.width + c, x[i]);
            load8<T, true>(p.gate + token * p.gate_stride + c, gs[i]);
            load8<T, true>(p.dy + token * p.width + c, d[i]);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                x[i][j] = live ? x[i][j] : 0.f;
                d[i][j] = live ? d[i][j] : 0.f;
                sum += x[i][j];
                sq = fmaf(x[i][j], x[i][j], sq);
            }
        }
        float mean = 0.f, scale;
        if (layer) {
            mean = wave_total<kWave>(sum) * inv_n;
            float var = 0.f;
#pragma unroll
            for (int i = 0; i < MAXC; ++i) {
                const bool live = (lane + i * kWave) * 8 < p.width;
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const float e = x[i][j] - mean;
                    var = live ? fmaf(e, e, var) : var;
                }
            }
            scale = rsqrtf(fmaf(wave_total<kWave>(var), inv_n, p.eps));
        } else {
            scale = rsqrtf(fmaf(wave_total<kWave>(sq), inv_n, p.eps));
        }
        // d <- d out / d (normalized x), and its projections on 1 and x
        float along = 0.f, level = 0.f;
#pragma unroll
        for (int i = 0; i < MAXC; ++i) {
            const int c = (lane + i * kWave) * 8;
            if (c >= p.width) continue;
            float wt[8], bs[8], dgate[8];
            param8<true>(p.weight, p.param_dtype, c, wt);
            if (layer) param8<true>(p.bias, p.param_dtype, c, bs);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const float n = (x[i][j] - mean) * scale, s = sigmoid_f(gs[i][j]);
                const float y = round_to<T>(layer ? fmaf(n, wt[j], bs[j]) : n * wt[j]);
                dgate[j] = d[i][j] * y * s * (1.f - s);
                const float dn = d[i][j] * s;
                dweight[i][j] = fmaf(dn, n, dweight[i][j]);
                dbias[i][j] += dn;
                x[i][j] = n;
                d[i][j] = dn * wt[j];
                along = fmaf(d[i][j], n, along);
                level += d[i][j];
            }
            store_row<8>(p.dgate + token * p.width + c, dgate);
        }
        along = wave_total<kWave>(along) * inv_n;
        level = layer ? wave_total<kWave>(level) * inv_n : 0.f;
#pragma unroll
        for (int i = 0; i < MAXC; ++i) {
            const int c = (lane + i * kWave) * 8;
            if (c >= p.width) continue;
            float dx[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) dx[j] = scale * (d[i][j] - level - x[i][j] * along);
            store_row<8>(p.draw + token * p.width + c, dx);
        }
    }
    extern __shared__ float red[];  // [waves][width]
    float *part = p.partials + int64_t(blockIdx.x) * 2 * p.width;
    for (int which = 0; which < (layer ? 2 : 1); ++which) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < MAXC; ++i) {
            const int c = (lane + i * kWave) * 8;
            if (c < p.width)
#pragma unroll
                for (int j = 0; j < 8; ++j) red[wave * p.width + c + j] = which ? dbias[i][j] : dweight[i][j];
        }
        __syncthreads();
        for (int c = threadIdx.x; c < p.width; c += blockDim.x) {
            float total = red[c];
            for (int w = 1; w < waves; ++w) total += red[w * p.width + c];
            part[which * p.width + c] = total;
        }
    }
}

// ------------------------------------------------------------------ router

// Softmax adjoint of a row's K selected pair sums, rounded as the values were,
// each added to the two factor scores it is the sum of: one thread per (row,
// score), the K terms in selection order.
template <typename T>
__global__ __launch_bounds__(256) void router_backward_kernel(const T *__restrict__ weights,
                                                              const int64_t *__restrict__ indices,
                                                              const T *__restrict__ grad, T *__restrict__ out,
                                                              int64_t rows, int j1, int j2, int k) {
    const int width = j1 + j2;
    const int64_t at = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (at >= rows * width) return;
    const int64_t row = at / width;
    const int col = int(at - row * width);
    float dot = 0.f, sum = 0.f;
    for (int j = 0; j < k; ++j) dot = fmaf(to_f32(weights[row * k + j]), to_f32(grad[row * k + j]), dot);
    for (int j = 0; j < k; ++j) {
        const int64_t bank = indices[row * k + j];
        const int first = int(bank / j2), second = int(bank - int64_t(first) * j2);
        const float d = round_to<T>(to_f32(weights[row * k + j]) * (to_f32(grad[row * k + j]) - dot));
        sum += (col < j1 ? first == col : second == col - j1) ? d : 0.f;
    }
    out[at] = from_f32<T>(sum);
}

}  // namespace
}  // namespace bdm

extern "C" int bdm_controller_backward(const bdm_controller_grad_args *a, void *stream) {
    using namespace bdm;
    if (!a) return fail(BDM_ERR_INVALID, "controller backward: null args");
    if (a->tokens <= 0 || a->tokens > INT32_MAX || a->heads <= 0 || a->head_width <= 0 || a->route_width <= 0)
        return fail(BDM_ERR_INVALID, "controller backward: bad geometry");
    const void *ptrs[] = {a->proj, a->f, a->dt_bias, a->grad_q, a->grad_k, a->grad_v, a->grad_b, a->grad_w, a->grad_g,
                          a->grad_read, a->grad_write, a->grad_proj, a->grad_f, a->grad_terms};
    for (const void *ptr : ptrs)
        if (!ptr || !aligned(ptr, 16)) return fail(BDM_ERR_INVALID, "controller backward: null or unaligned tensor");
    if (!aligned(a->grad_gate, 16)) return fail(BDM_ERR_INVALID, "controller backward: unaligned gate gradient");
    const int64_t cols[] = {a->q_col, a->k_col, a->v_col, a->b_col, a->w_col, a->read_col, a->write_col, a->gate_col,
                            a->proj_stride, a->f_stride, int64_t(a->heads) * a->head_width, a->route_width};
    for (int64_t c : cols)
        if (c < 0 || c % 8) return fail(BDM_ERR_UNSUPPORTED, "controller backward: columns must be multiples of 8");
    if (!a->a_log || a->ctrl_dtype != BDM_BF16 || (a->param_dtype != BDM_BF16 && a->param_dtype != BDM_F32))
        return fail(BDM_ERR_UNSUPPORTED, "controller backward: BF16 controllers, BF16 or FP32 parameters");
    ControllerGradParams<bf16_t> p{};
    auto in = [](const void *x) { return static_cast<const bf16_t *>(x); };
    p.proj = in(a->proj), p.f = in(a->f);
    p.a_log = a->a_log, p.dt_bias = a->dt_bias;
    p.dq = in(a->grad_q), p.dk = in(a->grad_k), p.dv = in(a->grad_v), p.db = in(a->grad_b), p.dw = in(a->grad_w);
    p.dread = in(a->grad_read), p.dwrite = in(a->grad_write), p.dgate = in(a->grad_gate);
    p.dg = a->grad_g;
    p.dproj = static_cast<bf16_t *>(a->grad_proj), p.df = static_cast<bf16_t *>(a->grad_f);
    p.terms = a->grad_terms;
    p.proj_stride = a->proj_stride, p.f_stride = a->f_stride;
    p.q_col = a->q_col, p.k_col = a->k_col, p.v_col = a->v_col, p.b_col = a->b_col, p.w_col = a->w_col;
    p.read_col = a->read_col, p.write_col = a->write_col, p.gate_col = a->gate_col;
    p.heads = a->heads, p.hv = a->head_width, p.route_width = a->route_width;
    p.param_dtype = a->param_dtype, p.qk_norm = a->qk_norm;
    const unsigned blocks = unsigned(a->tokens);
    hipStream_t s = as_stream(stream);
    switch (a->bank_size) {
        case 8: controller_backward_kernel<bf16_t, 8><<<blocks, 256, 0, s>>>(p); break;
        case 16: controller_backward_kernel<bf16_t, 16><<<blocks, 256, 0, s>>>(p); break;
        case 32: controller_backward_kernel<bf16_t, 32><<<blocks, 256, 0, s>>>(p); break;
        default: return fail(BDM_ERR_UNSUPPORTED, "controller backward: bank_size %d", a->bank_size);
    }
    return check_launch("controller_backward_kernel");
}

extern "C" int64_t bdm_output_backward_partials(int64_t tokens) {
    return tokens <= 0 ? 0 : (tokens + bdm::kOutputRows - 1) / bdm::kOutputRows;
}

extern "C" int bdm_output_backward(const bdm_output_grad_args *a, void *stream) {
    using namespace bdm;
    if (!a) return fail(BDM_ERR_INVALID, "output backward: null args");
    if (a->tokens <= 0 || a->width <= 0 || a->width % 8 || a->gate_stride % 8)
        return fail(BDM_ERR_INVALID, "output backward: bad geometry");
    if (a->width > 4096) return fail(BDM_ERR_UNSUPPORTED, "output backward: width %d > 4096", a->width);
    const void *ptrs[] = {a->raw, a->gate, a->grad_out, a->norm_weight, a->grad_raw, a->grad_gate, a->partials};
    for (const void *ptr : ptrs)
        if (!ptr || !aligned(ptr, 16)) return fail(BDM_ERR_INVALID, "output backward: null or unaligned tensor");
    if (a->norm_kind == 1 && (!a->norm_bias || !aligned(a->norm_bias, 16)))
        return fail(BDM_ERR_INVALID, "output backward: layer norm needs an aligned bias");
    if (a->ctrl_dtype != BDM_BF16 || (a->param_dtype != BDM_BF16 && a->param_dtype != BDM_F32))
        return fail(BDM_ERR_UNSUPPORTED, "output backward: BF16 rows, BF16 or FP32 parameters");
    OutputGradParams<bf16_t> p{};
    p.raw = static_cast<const bf16_t *>(a->raw), p.gate = static_cast<const bf16_t *>(a->gate);
    p.dy = static_cast<const bf16_t *>(a->grad_out);
    p.weight = a->norm_weight, p.bias = a->norm_bias;
    p.draw = static_cast<bf16_t *>(a->grad_raw), p.dgate = static_cast<bf16_t *>(a->grad_gate);
    p.partials = a->partials;
    p.tokens = a->tokens, p.gate_stride = a->gate_stride;
    p.width = a->width, p.param_dtype = a->param_dtype, p.norm_kind = a->norm_kind, p.eps = a->eps;
    const int64_t blocks = bdm_output_backward_partials(a->tokens);
    if (blocks > INT32_MAX) return fail(BDM_ERR_UNSUPPORTED, "output backward: too many tokens");
    const size_t lds = size_t(4) * size_t(a->width) * sizeof(float);
    const int chunks = (a->width / 8 + kWave - 1) / kWave;
    hipStream_t s = as_stream(stream);
    if (chunks <= 1) output_backward_kernel<bf16_t, 1><<<unsigned(blocks), 256, lds, s>>>(p);
    else if (chunks <= 2) output_backward_kernel<bf16_t, 2><<<unsigned(blocks), 256, lds, s>>>(p);
    else if (chunks <= 4) output_backward_kernel<bf16_t, 4><<<unsigned(blocks), 256, lds, s>>>(p);
    else output_backward_kernel<bf16_t, 8><<<unsigned(blocks), 256, lds, s>>>(p);
    return check_launch("output_backward_kernel");
}

extern "C" int bdm_router_backward(const void *weights, const int64_t *indices, const void *grad_weights, void *grad_scores,
                                   int64_t rows, int32_t factor_first, int32_t factor_second, int32_t selected,
                                   int32_t dtype, void *stream) {
    using namespace bdm;
    if (rows < 0 || factor_first <= 0 || factor_second <= 0 || selected <= 0)
        return fail(BDM_ERR_INVALID, "router backward: bad geometry");
    if (rows == 0) return BDM_OK;
    if (!weights || !indices || !grad_weights || !grad_scores)
        return fail(BDM_ERR_INVALID, "router backward: null pointer");
    const int64_t blocks = (rows * (int64_t(factor_first) + factor_second) + 255) / 256;
    if (blocks > INT32_MAX) return fail(BDM_ERR_UNSUPPORTED, "router backward: too many rows");
    hipStream_t s = as_stream(stream);
    if (dtype == BDM_BF16)
        router_backward_kernel<bf16_t><<<unsigned(blocks), 256, 0, s>>>(
            static_cast<const bf16_t *>(weights), indices, static_cast<const bf16_t *>(grad_weights),
            static_cast<bf16_t *>(grad_scores), rows, factor_first, factor_second, selected);
    else if (dtype == BDM_F32)
        router_backward_kernel<float><<<unsigned(blocks), 256, 0, s>>>(
            static_cast<const float *>(weights), indices, static_cast<const float *>(grad_weights),
            static_cast<float *>(grad_scores), rows, factor_first, factor_second, selected);
    else
        return fail(BDM_ERR_INVALID, "router backward: dtype %d", dtype);
    return check_launch("router_backward_kernel");
}

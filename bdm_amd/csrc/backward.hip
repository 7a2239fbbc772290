// Backward of the routed GDN2 bank recurrence and the token-level VJP.
//
// Reference: _role_backward (role_bank_kernel.py:76-150, launched by
// backward() at :205-228), RoutedUpdate.backward (routed_update.py:31-49:
// the decay term of d(ww) and dg scaled by p) and _vjp
// (role_bank_dispatch.py:76-132, with its BF16 rounding points).
//
// Per write event the adjoint dM (S x v) of the state after the event gives
//   du = dM^T k;  U = dM u;  X = hd du;  P = rowsum(dM o hd)
//   dM <- (dM - a du^T) o decay                (role_bank_kernel.py:128-138)
// and per read event dq = scale M dy, dM += scale eq dy^T (:141-143).  U, X
// and P (S values each) are stored per event; the token kernel forms
// dk = U - eb X, db = -k X, dg = P - a X from them and the event's operands.
//
// chunk_backward_kernel (S = 8, replay interval 16): one wave per (segment,
// head, column tile); a lane owns 2 value columns and all 8 rows.  Chunks of
// 16 events are visited in reverse.  The chunk's states are rebuilt exactly
// from its snapshot by the forward's write update, in two halves of 8 events:
// the states before events 8..15 are kept in registers while the second half
// is differentiated, then those before events 0..7.  Per event operands (the
// write's k, decay, a rows and bf(w p), v columns; the read's eq*scale row
// and dy columns) are staged in LDS one chunk ahead: the next chunk's loads
// are issued before the current chunk's last half is differentiated.  The
// S-wide column reductions use permlane swaps and DPP row sums
// (reduce-scatter: each output ends in one lane, no LDS round trip).
//
// staged_backward_kernel: every other S <= 32 and interval of 4, 8 or 16.
//
// token_grad_kernel: one workgroup per token, one wave per head.  Lane
// (j, r) = (lane / 8, lane % 8) handles route slot j and state row r of the
// S-side gradients; lanes own 2 value columns for dv, dw.  The token's KW
// write events and KR read events are folded in route order with the
// reference's rounding (role_bank_dispatch.py:99-131); route-weight
// gradients add the heads' contributions in head order in FP32.
// token_vjp_kernel: the same for shapes outside that kernel's limits.
#include <algorithm>
#include <type_traits>

#include "bdm_common.h"
#include "recurrence_ops.h"
#include "segment_order.h"

namespace bdm {
namespace {

constexpr int kLanes = 64;

template <typename T>
struct BackwardParams {
    const T *q, *k, *b;
    const float *g;
    const T *v, *w;
    const T *ww, *rw;
    const int64_t *order, *cu;
    const void *initial;
    const void *snap;
    const T *dy;
    float *du;      // [NT*KW, H, v]
    float *wpart;   // [tiles, NT*KW, H, 3, S]: U, X, P of each write slot
    float *rpart;   // [tiles, NT*KR, H, S]: dq of each read slot
    const int4 *meta;  // [E]: token, route slot, is_read, route weight (FP32 bits)
    float *dinit;   // [batch, J, H, S, v]
    int64_t init_bstride, nt;
    int heads, s_real, width, banks, kw, kr, tiles;
    int k_shift;  // log2 of KW and KR when both are that power of two, else -1 (route -> token by shift)
    int init_dtype, snap_dtype, routed_decay, rounding;
    int xcd_remap;
    float scale;
    // chunk kernel: each XCD range's segments longest first
    // (segment_order_kernel), in rounds of order_gpr (head, tile) items;
    // null keeps bank order
    const int *seg_order;
    int order_gpr;
};

// ------------------------------------------------- S = 8, replay interval 16

template <int CTRL>
__device__ __forceinline__ float dpp_add(float x) {
    return x + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xF, 0xF,
                                                                     false));
}

// x of the lane CTRL (a DPP row_shr / row_shl) names inside the 16-lane row,
// 1 where that lane lies outside the row.
template <int CTRL>
__device__ __forceinline__ float row_shift(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, 1.f),
                                                                 __builtin_bit_cast(int, x), CTRL, 0xF, 0xF, false));
}

// x * (x of the lane CTRL selects within the row), or x where that lane lies
// outside the row: one v_mul_f32 with a DPP source and bound_ctrl off (the
// lane without a source does not write).  CTRL: 0x111/0x112/0x114/0x118 are
// row_shr 1/2/4/8, 0x101/0x102/0x104/0x108 row_shl 1/2/4/8.  The s_nop gives
// the 2 wait states a DPP read of a VGPR needs after a VALU write of it.
template <int CTRL>
__device__ __forceinline__ float row_mul_step(float x) {
#define BDM_DPP_MUL(SEL) asm volatile("s_nop 1\n\tv_mul_f32_dpp %0, %0, %0 " SEL " row_mask:0xf bank_mask:0xf" : "+v"(x))
    if constexpr (CTRL == 0x111) BDM_DPP_MUL("row_shr:1");
    else if constexpr (CTRL == 0x112) BDM_DPP_MUL("row_shr:2");
    else if constexpr (CTRL == 0x114) BDM_DPP_MUL("row_shr:4");
    else if constexpr (CTRL == 0x118) BDM_DPP_MUL("row_shr:8");
    else if constexpr (CTRL == 0x101) BDM_DPP_MUL("row_shl:1");
    else if constexpr (CTRL == 0x102) BDM_DPP_MUL("row_shl:2");
    else if constexpr (CTRL == 0x104) BDM_DPP_MUL("row_shl:4");
    else if constexpr (CTRL == 0x108) BDM_DPP_MUL("row_shl:8");
    else static_assert(CTRL == 0x111, "row_mul_step: unsupported DPP control");
#undef BDM_DPP_MUL
    return x;
}

// Total of a 16-lane row in every lane of the row.
__device__ __forceinline__ float row_total(float x) {
    x = dpp_add<0xB1>(x);      // quad_perm [1,0,3,2]
    x = dpp_add<0x4E>(x);      // quad_perm [2,3,0,1]
    x = dpp_add<0x141>(x);     // row_half_mirror: quads 0 <-> 1, 2 <-> 3
    return dpp_add<0x140>(x);  // row_mirror: halves of the row
}

// Sums each of N values over the 64 lanes of the wave.  Value o = (N/4) * row
// + i (row = lane / 16) ends in the lanes of that row at position
// lane % 16 = i < N/4, which return it; other lanes return a partial sum.
template <int N>
__device__ __forceinline__ float reduce_scatter(const float (&x)[N], int lane) {
    static_assert(N % 4 == 0, "N");
    float y[N / 2];
#pragma unroll
    for (int i = 0; i < N / 2; ++i) y[i] = half_pair_sum(x[i], x[i + N / 2]);
    float z[N / 4];
#pragma unroll
    for (int i = 0; i < N / 4; ++i) z[i] = row_total(row_pair_sum(y[i], y[i + N / 4]));
    const int pos = lane & 15;
    float out = z[0];
#pragma unroll
    for (int i = 1; i < N / 4; ++i) out = pos == i ? z[i] : out;
    // computed in every lane: keeps the DPP adds fused when the caller stores
    // from a subset of lanes
    asm volatile("" : "+v"(out));
    return out;
}

// Sums of N values over the lane's 32-lane half partners and row partners: the
// first two steps of reduce_scatter.  z[i] of row j (lane / 16) is a 16-lane
// partial of value (N / 4) j + i.
template <int N>
__device__ __forceinline__ void sum_rows(const float (&x)[N], float (&z)[N / 4]) {
    float y[N / 2];
#pragma unroll
    for (int i = 0; i < N / 2; ++i) y[i] = half_pair_sum(x[i], x[i + N / 2]);
#pragma unroll
    for (int i = 0; i < N / 4; ++i) z[i] = row_pair_sum(y[i], y[i + N / 4]);
}

// Totals over 16-lane rows of six values in 13 additions where each value's own
// row_total takes 4 (24): a DPP addition that writes only some of a row's four
// banks (of 4 lanes) leaves room in the others for the next value.  A lane at
// position t of its row returns, for t % 8 = 0, 4 and 1, the total of
// a[0], a[1] and a[2] (t < 8) or of b[0], b[1] and b[2].  chunk_backward_kernel:
// 566 -> 546 us at 8,192 tokens, H8 v128, 1,058 -> 1,040 with one head of 2,048
// columns.  The order of the
// instructions and the s_nop give the 2 wait states a DPP read of a VGPR needs
// after a VALU write of it.
__device__ __forceinline__ float row_totals6(float (&a)[3], const float (&b)[3], int lane) {
    asm volatile("s_nop 1\n\t"
                 "v_add_f32_dpp %0, %0, %0 row_mirror row_mask:0xf bank_mask:0x3\n\t"
                 "v_add_f32_dpp %0, %3, %3 row_mirror row_mask:0xf bank_mask:0xc\n\t"
                 "v_add_f32_dpp %1, %1, %1 row_mirror row_mask:0xf bank_mask:0x3\n\t"
                 "v_add_f32_dpp %1, %4, %4 row_mirror row_mask:0xf bank_mask:0xc\n\t"
                 "v_add_f32_dpp %2, %2, %2 row_mirror row_mask:0xf bank_mask:0x3\n\t"
                 "v_add_f32_dpp %2, %5, %5 row_mirror row_mask:0xf bank_mask:0xc\n\t"
                 "v_add_f32_dpp %0, %0, %0 row_half_mirror row_mask:0xf bank_mask:0x5\n\t"
                 "v_add_f32_dpp %0, %1, %1 row_half_mirror row_mask:0xf bank_mask:0xa\n\t"
                 "v_add_f32_dpp %2, %2, %2 row_half_mirror row_mask:0xf bank_mask:0xf\n\t"
                 "s_nop 0\n\t"
                 "v_add_f32_dpp %0, %0, %0 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
                 "v_add_f32_dpp %2, %2, %2 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
                 "s_nop 0\n\t"
                 "v_add_f32_dpp %0, %0, %0 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
                 "v_add_f32_dpp %2, %2, %2 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf"
                 : "+&v"(a[0]), "+&v"(a[1]), "+&v"(a[2])
                 : "v"(b[0]), "v"(b[1]), "v"(b[2]));
    return (lane & 3) == 0 ? a[0] : a[2];
}

// The same of two values: lanes 0..7 of a row return a's total, 8..15 b's.
__device__ __forceinline__ float row_totals2(float a, float b) {
    asm volatile("s_nop 1\n\t"
                 "v_add_f32_dpp %0, %0, %0 row_mirror row_mask:0xf bank_mask:0x3\n\t"
                 "v_add_f32_dpp %0, %1, %1 row_mirror row_mask:0xf bank_mask:0xc\n\t"
                 "s_nop 1\n\t"
                 "v_add_f32_dpp %0, %0, %0 row_half_mirror row_mask:0xf bank_mask:0xf\n\t"
                 "s_nop 1\n\t"
                 "v_add_f32_dpp %0, %0, %0 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
                 "s_nop 1\n\t"
                 "v_add_f32_dpp %0, %0, %0 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf"
                 : "+&v"(a)
                 : "v"(b));
    return a;
}

// One entry per event of the packed order: token, route slot, is_read and
// the route weight (FP32 bits), shared by every head.
template <typename T>
__global__ __launch_bounds__(256) void event_meta_kernel(const int64_t *order, int64_t events, int64_t write_events,
                                                         int kw, int kr, const T *ww, const T *rw, int4 *meta) {
    const int64_t e = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (e >= events) return;
    int64_t o = order[e];
    o = o < 0 ? 0 : (o >= events ? events - 1 : o);
    const bool rd = o >= write_events;
    const int64_t route = rd ? o - write_events : o;
    const int64_t token = rd ? route / kr : route / kw;
    const float weight = to_f32(rd ? rw[route] : ww[route]);
    meta[e] = make_int4(int(token), int(route), rd ? 1 : 0, __float_as_int(weight));
}

// Lane e's address, uniform over the wave.
__device__ __forceinline__ const char *lane_ptr(uint64_t x, int e) {
    const uint32_t lo = __builtin_amdgcn_readlane(uint32_t(x), e), hi = __builtin_amdgcn_readlane(uint32_t(x >> 32), e);
    return reinterpret_cast<const char *>(uint64_t(hi) << 32 | lo);
}

template <typename T, typename SNAP>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void chunk_backward_kernel(
    BackwardParams<T> p) {
    constexpr int S = 8, CPL = 2, C = 16, HALF = 8;
    // Per-event operand row (64 floats).  Write: the adjoint's k*sigma,
    // erase coefficient a*decay*s, update a/sigma, replay k/s', the output
    // scales of U, X, P and the decay; read: eq*scale/sigma and dq's scale.
    constexpr int kKey = 0, kErase = 8, kUpd = 16, kRep = 24, kScale = 32, kDecay = 56;
    using P2 = Pair<T>;
    using Raw = typename P2::raw;
    using SnapRaw = typename Pair<SNAP>::raw;
    struct ColSlot {
        Raw a, b;  // write: v, bf(w p); read: dy, unused
    };
    struct Staged {
        Raw a[C], b[C];
        Raw kq, bb;
        float2 g;
        SnapRaw m0[S];  // snapshot rows (chunks > 0)
    };
    __shared__ int4 s_meta[2][C];
    __shared__ float4 s_rows[C][16];
    __shared__ ColSlot s_cols[C][kLanes];
    __shared__ float2 s_m0[S][kLanes];  // the chunk's start state, lane's column pair per row
    __shared__ float s_fold[S];         // product of the chunk's decays per row (lazy chunks) or 1
    __shared__ int s_eager;

    int seg, head, tile;
    block_item(p, seg, head, tile);
    const int bank = seg % p.banks;
    const int64_t bidx = seg / p.banks;
    const int lane = threadIdx.x;
    const int col0 = (tile * kLanes + lane) * CPL;
    const bool live = col0 < p.width;
    const int colc = live ? col0 : p.width - CPL;  // lanes past the width load a valid pair and zero it
    const int64_t start = p.cu[seg], end = p.cu[seg + 1];
    const int count = int((end - start + C - 1) / C);
    const uint32_t hw = uint32_t(p.heads) * uint32_t(p.width);
    const int lane_col = head * p.width + colc;  // offset of the lane's pair in a [token] row of H*v
    // event-uniform bases: x[slot] + per-lane offset
    float *du_lane = p.du + head * p.width + col0;
    float *wp_tile = p.wpart + (int64_t(tile) * p.nt * p.kw * p.heads + head) * 3 * S;
    float *rp_tile = p.rpart + (int64_t(tile) * p.nt * p.kr * p.heads + head) * S;

    auto chunk_len = [&](int c) { return int(min(int64_t(C), end - (start + int64_t(c) * C))); };
    auto load_meta = [&](int c) {
        const int len = chunk_len(c);
        return p.meta[start + int64_t(c) * C + (lane < len ? lane : len - 1)];
    };
    auto store_meta = [&](int c, const int4 &m) {
        if (lane < C) s_meta[c & 1][lane] = m;
    };
    // Loads of chunk c's operands and start state (its meta is in LDS).  Lane e
    // (mod C) forms the row addresses of event e, each event takes them with
    // v_readlane as its loads' scalar base, where each event waited for its LDS
    // read and formed both addresses in scalar instructions (546 -> 510 us at
    // 8,192 tokens, H8 v128, 1,040 -> 974 with one head of 2,048 columns).
    auto issue_stage = [&](int c, Staged &sg) {
        const int len = chunk_len(c);
        const int ev = lane & (C - 1);
        const int4 m = s_meta[c & 1][ev < len ? ev : len - 1];
        const uint64_t row = uint64_t(uint32_t(m.x)) * hw;
        const uint64_t ra = reinterpret_cast<uint64_t>((m.z ? p.dy : p.v) + row);
        const uint64_t rb = reinterpret_cast<uint64_t>((m.z ? p.dy : p.w) + row);
        const uint32_t byte = uint32_t(lane_col) * uint32_t(sizeof(T));
#pragma unroll
        for (int e = 0; e < C; ++e) {
            sg.a[e] = P2::load(reinterpret_cast<const T *>(lane_ptr(ra, e) + byte));
            sg.b[e] = P2::load(reinterpret_cast<const T *>(lane_ptr(rb, e) + byte));
        }
        {
            const int rp = (lane >> 4) * 2;
            const int64_t at = (int64_t(m.x) * p.heads + head) * S + rp;
            sg.kq = P2::load((m.z ? p.q : p.k) + at);
            sg.bb = P2::load(p.b + at);
            sg.g = *reinterpret_cast<const float2 *>(p.g + at);
        }
        if (c > 0) {
            const SNAP *snap = static_cast<const SNAP *>(p.snap) +
                               (((start + int64_t(c) * C) / C - 1) * p.heads + head) * S * p.width + colc;
#pragma unroll
            for (int r = 0; r < S; ++r) sg.m0[r] = Pair<SNAP>::load(snap + r * p.width);
        }
    };
    // Operand rows, columns and the start state of chunk c into LDS.
    auto finish_stage = [&](int c, const Staged &sg) {
        const int len = chunk_len(c);
        // lane = 16 j + e holds rows 2j, 2j+1 of event e: the scans over a
        // chunk's events run inside 16-lane rows (DPP row shifts)
        const int e = lane & (C - 1), rp = (lane >> 4) * 2;
        const int4 m = s_meta[c & 1][e < len ? e : len - 1];
#pragma unroll
        for (int i = 0; i < C; ++i) {
            ColSlot cs;  // a read's b is not used
            cs.a = live ? sg.a[i] : P2::zero();
            cs.b = live ? P2::scaled(sg.b[i], __int_as_float(__builtin_amdgcn_readlane(m.w, i))) : P2::zero();
            s_cols[i][lane] = cs;
        }
        {
            const bool valid = e < len;
            const bool wr = valid && m.z == 0;
            const float pw = __int_as_float(m.w);
            const float x[2] = {P2::lo(sg.kq), P2::hi(sg.kq)};  // k of a write, q of a read
            const float bv[2] = {P2::lo(sg.bb), P2::hi(sg.bb)};
            const float gv[2] = {sg.g.x, sg.g.y};
            float d[2], a[2], pre[2], suf[2], pre_x[2], suf_x[2];
            bool bad = false;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                // decay = exp(g p), a = bf(b p) k (prepare_write_rows); 1 for reads
                d[i] = wr ? __expf(p.routed_decay ? gv[i] * pw : gv[i]) : 1.f;
                a[i] = round_to<T>(bv[i] * pw) * x[i];
                // inclusive prefix and suffix products of the decays over the chunk's events
                pre[i] = row_mul_step<0x118>(row_mul_step<0x114>(row_mul_step<0x112>(row_mul_step<0x111>(d[i]))));
                suf[i] = row_mul_step<0x108>(row_mul_step<0x104>(row_mul_step<0x102>(row_mul_step<0x101>(d[i]))));
                pre_x[i] = row_shift<0x111>(pre[i]);
                suf_x[i] = row_shift<0x101>(suf[i]);
                const float lo = 0x1p-40f, hi = 0x1p40f;
                bad |= !(pre[i] >= lo && pre[i] <= hi && suf[i] >= lo && suf[i] <= hi);
            }
            // Lazy chunk: state diag(s) Mh with s = the decays of the chunk's earlier
            // writes, adjoint diag(sigma) dMh with sigma = those of its later writes.
            // Eager chunk (a product out of range): s = sigma = 1 and both are
            // multiplied by the decay after each write.
            const bool eager = __ballot(bad) != 0;
            float *row = reinterpret_cast<float *>(&s_rows[e][0]);
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int r = rp + i;
                const float s = eager ? 1.f : pre_x[i];                // before the event
                const float s1 = eager ? fmaxf(d[i], 0x1p-40f) : pre[i];  // after a write
                const float sg_ = eager ? 1.f : suf_x[i];
                const float inv_sg = __builtin_amdgcn_rcpf(sg_);
                if (m.z) {
                    const float eqs = round_to<T>(x[i] * pw) * p.scale;
                    row[kKey + r] = eqs * inv_sg;
                    row[kScale + r] = p.scale * s;
                } else {
                    row[kKey + r] = x[i] * sg_;
                    row[kErase + r] = a[i] * d[i] * s;
                    row[kUpd + r] = a[i] * inv_sg;
                    row[kRep + r] = x[i] * __builtin_amdgcn_rcpf(s1);
                    row[kScale + r] = sg_;
                    row[kScale + S + r] = d[i] * s;
                    row[kScale + 2 * S + r] = d[i] * s * sg_;
                    row[kDecay + r] = s1;
                }
                if (e == 0) s_fold[r] = eager ? 1.f : suf[i];
            }
            if (lane == 0) s_eager = eager ? 1 : 0;
        }
        float m0[S][CPL];
        if (c > 0) {
#pragma unroll
            for (int r = 0; r < S; ++r) {
                m0[r][0] = live ? Pair<SNAP>::lo(sg.m0[r]) : 0.f;
                m0[r][1] = live ? Pair<SNAP>::hi(sg.m0[r]) : 0.f;
            }
        } else {
            // the segment's initial state (rounded to BF16 under the rounding policy)
            const int64_t off = bidx * p.init_bstride + (int64_t(bank) * p.heads + head) * S * p.width + colc;
            float lo[S], hi[S];
            if (p.init_dtype == BDM_BF16) {
                uint32_t x[S];
#pragma unroll
                for (int r = 0; r < S; ++r)
                    x[r] = Pair<bf16_t>::load(static_cast<const bf16_t *>(p.initial) + off + r * p.width);
#pragma unroll
                for (int r = 0; r < S; ++r) lo[r] = Pair<bf16_t>::lo(x[r]), hi[r] = Pair<bf16_t>::hi(x[r]);
            } else {
                float2 x[S];
#pragma unroll
                for (int r = 0; r < S; ++r)
                    x[r] = Pair<float>::load(static_cast<const float *>(p.initial) + off + r * p.width);
#pragma unroll
                for (int r = 0; r < S; ++r) {
                    lo[r] = x[r].x, hi[r] = x[r].y;
                    if (p.rounding) round_pair<bf16_t>(lo[r], hi[r]);
                }
            }
#pragma unroll
            for (int r = 0; r < S; ++r) {
                m0[r][0] = live ? lo[r] : 0.f;
                m0[r][1] = live ? hi[r] : 0.f;
            }
        }
#pragma unroll
        for (int r = 0; r < S; ++r) s_m0[r][lane] = make_float2(m0[r][0], m0[r][1]);
    };
    auto load_m0 = [&](float (&m)[S][CPL]) {
#pragma unroll
        for (int r = 0; r < S; ++r) {
            const float2 x = s_m0[r][lane];
            m[r][0] = x.x;
            m[r][1] = x.y;
        }
    };
    auto rows8 = [&](int e, int at, float (&x)[S]) {
        const float4 lo = s_rows[e][at / 4], hi = s_rows[e][at / 4 + 1];
        x[0] = lo.x, x[1] = lo.y, x[2] = lo.z, x[3] = lo.w, x[4] = hi.x, x[5] = hi.y, x[6] = hi.z, x[7] = hi.w;
    };
    // Replay of write e: u = bf(w p) v - sum_r (a decay s)_r Mh_r ; Mh += (k / s') u.
    auto apply = [&](int e, float (&m)[S][CPL]) {
        float ce[S], kt[S];
        rows8(e, kErase, ce);
        rows8(e, kRep, kt);
        const ColSlot cs = s_cols[e][lane];
        const float v[CPL] = {P2::lo(cs.a), P2::hi(cs.a)}, ew[CPL] = {P2::lo(cs.b), P2::hi(cs.b)};
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
            float erase = 0.f;
#pragma unroll
            for (int r = 0; r < S; ++r) erase = fmaf(ce[r], m[r][c], erase);
            const float u = fmaf(ew[c], v[c], -erase);
#pragma unroll
            for (int r = 0; r < S; ++r) m[r][c] = fmaf(kt[r], u, m[r][c]);
        }
    };
    // Eager chunks: multiply by the decay after a write.
    auto fold = [&](int e, float (&m)[S][CPL]) {
        float dd[S];
        rows8(e, kDecay, dd);
#pragma unroll
        for (int r = 0; r < S; ++r)
#pragma unroll
            for (int c = 0; c < CPL; ++c) m[r][c] *= dd[r];
    };

    float dm[S][CPL];
#pragma unroll
    for (int r = 0; r < S; ++r)
#pragma unroll
        for (int c = 0; c < CPL; ++c) dm[r][c] = 0.f;

    // The output of the lane in row_totals6's layout (value 3 j + i of U, X, P by
    // rows 4 g .. 4 g + 3: j the 16-lane row, i = 0, 1, 2 at positions 0, 4, 1 of
    // its half g) and in row_totals2's (rows 2 j and 2 j + 1 of dq).
    const int w_pos = lane & 7, w_out = 3 * (lane >> 4) + (w_pos == 0 ? 0 : (w_pos == 4 ? 1 : 2));
    const int w_at = (w_out >> 2) * S + 4 * ((lane >> 3) & 1) + (w_out & 3);
    const bool w_mine = w_pos == 0 || w_pos == 4 || w_pos == 1;
    const int r_at = 2 * (lane >> 4) + ((lane >> 3) & 1);

    // Adjoint of write e, pre-event state st = diag(s) Mh, dm = diag(sigma) dMh:
    //   du = dMh^T (k sigma); u = x - Mh^T (a decay s)
    //   U = sigma (dMh u); X = decay s (Mh du); P = decay s sigma rowsum(dMh o Mh)
    //   dMh -= (a / sigma) du^T                      (role_bank_kernel.py:128-138)
    auto write_back = [&](int e, int slots, const float (&st)[S][CPL]) {
        float kk[S], ce[S], au[S];
        rows8(e, kKey, kk);
        rows8(e, kErase, ce);
        rows8(e, kUpd, au);
        const ColSlot cs = s_cols[e][lane];
        const float v[CPL] = {P2::lo(cs.a), P2::hi(cs.a)}, ew[CPL] = {P2::lo(cs.b), P2::hi(cs.b)};
        float u[CPL], du[CPL];
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
            float erase = 0.f, acc = 0.f;
#pragma unroll
            for (int r = 0; r < S; ++r) {
                erase = fmaf(ce[r], st[r][c], erase);
                acc = fmaf(dm[r][c], kk[r], acc);
            }
            u[c] = fmaf(ew[c], v[c], -erase);
            du[c] = acc;
        }
        const uint32_t slot = uint32_t(__builtin_amdgcn_readlane(slots, e));
        if (live) *reinterpret_cast<float2 *>(du_lane + uint64_t(slot) * hw) = make_float2(du[0], du[1]);
        float *wp = wp_tile + uint64_t(slot) * uint32_t(p.heads * 3 * S);
        // rows 0..3, then 4..7: red = U[4], X[4], P[4] of the group
        float z[2][3];
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            float red[12];
#pragma unroll
            for (int i = 0; i < 12; ++i) red[i] = 0.f;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int r = 4 * g + i;
#pragma unroll
                for (int c = 0; c < CPL; ++c) {
                    red[i] = fmaf(dm[r][c], u[c], red[i]);
                    red[4 + i] = fmaf(st[r][c], du[c], red[4 + i]);
                    red[8 + i] = fmaf(dm[r][c], st[r][c], red[8 + i]);
                    dm[r][c] = fmaf(-au[r], du[c], dm[r][c]);
                }
            }
            sum_rows<12>(red, z[g]);
        }
        const float o = row_totals6(z[0], z[1], lane) * reinterpret_cast<const float *>(&s_rows[e][0])[kScale + w_at];
        if (w_mine) wp[w_at] = o;
    };
    // Adjoint of read e with state st = diag(s) Mh: dq = scale s (Mh dy); dMh += (eq scale / sigma) dy^T.
    auto read_back = [&](int e, int slots, const float (&st)[S][CPL]) {
        float eq[S];
        rows8(e, kKey, eq);
        const ColSlot cs = s_cols[e][lane];
        const float dy[CPL] = {P2::lo(cs.a), P2::hi(cs.a)};
        float red[S];
#pragma unroll
        for (int r = 0; r < S; ++r) {
            red[r] = 0.f;
#pragma unroll
            for (int c = 0; c < CPL; ++c) red[r] = fmaf(st[r][c], dy[c], red[r]);
        }
#pragma unroll
        for (int r = 0; r < S; ++r)
#pragma unroll
            for (int c = 0; c < CPL; ++c) dm[r][c] = fmaf(eq[r], dy[c], dm[r][c]);
        const uint32_t slot = uint32_t(__builtin_amdgcn_readlane(slots, e));
        float z[S / 4];
        sum_rows<S>(red, z);
        const float o = row_totals2(z[0], z[1]) * reinterpret_cast<const float *>(&s_rows[e][0])[kScale + r_at];
        if ((lane & 7) == 0) rp_tile[uint64_t(slot) * uint32_t(p.heads * S) + r_at] = o;
    };

    if (count > 0) {
        store_meta(count - 1, load_meta(count - 1));
        int4 prev = make_int4(0, 0, 0, 0);
        if (count > 1) prev = load_meta(count - 2);
        __syncthreads();
        Staged sg;
        issue_stage(count - 1, sg);
        if (count > 1) store_meta(count - 2, prev);
        __syncthreads();
        finish_stage(count - 1, sg);
    }

#pragma unroll 1
    for (int c = count - 1; c >= 0; --c) {
        __syncthreads();
        const int len = chunk_len(c);
        const int4 mine = s_meta[c & 1][lane & (C - 1)];
        const uint32_t wmask = uint32_t(__ballot(lane < len && mine.z == 0)) & 0xffffu;
        const uint32_t rmask = uint32_t(__ballot(lane < len && mine.z != 0)) & 0xffffu;
        const uint32_t fmask = __builtin_amdgcn_readfirstlane(s_eager) ? wmask : 0u;
        float st[HALF][S][CPL];
        if (len > HALF) {
            float m[S][CPL];
            load_m0(m);
#pragma unroll
            for (int e = 0; e < C - 1; ++e) {
                if (e >= HALF) {
#pragma unroll
                    for (int r = 0; r < S; ++r)
#pragma unroll
                        for (int cc = 0; cc < CPL; ++cc) st[e - HALF][r][cc] = m[r][cc];
                }
                if (wmask & (1u << e)) apply(e, m);
                if (fmask & (1u << e)) fold(e, m);
            }
#pragma unroll
            for (int r = 0; r < S; ++r)
#pragma unroll
                for (int cc = 0; cc < CPL; ++cc) st[HALF - 1][r][cc] = m[r][cc];
#pragma unroll
            for (int e = C - 1; e >= HALF; --e) {
                if (wmask & (1u << e)) write_back(e, mine.y, st[e - HALF]);
                else if (rmask & (1u << e)) read_back(e, mine.y, st[e - HALF]);
                if (fmask & (1u << e)) fold(e, dm);
            }
        }
        {
            float m[S][CPL];
            load_m0(m);
#pragma unroll
            for (int e = 0; e < HALF; ++e) {
#pragma unroll
                for (int r = 0; r < S; ++r)
#pragma unroll
                    for (int cc = 0; cc < CPL; ++cc) st[e][r][cc] = m[r][cc];
                if (e + 1 < HALF) {
                    if (wmask & (1u << e)) apply(e, m);
                    if (fmask & (1u << e)) fold(e, m);
                }
            }
        }
        // the next chunk's loads, in flight while events 7..0 are differentiated
        int4 meta2 = make_int4(0, 0, 0, 0);
        Staged sg;
        if (c >= 2) meta2 = load_meta(c - 2);
        if (c >= 1) issue_stage(c - 1, sg);
#pragma unroll
        for (int e = HALF - 1; e >= 0; --e) {
            if (wmask & (1u << e)) write_back(e, mine.y, st[e]);
            else if (rmask & (1u << e)) read_back(e, mine.y, st[e]);
            if (fmask & (1u << e)) fold(e, dm);
        }
        // the adjoint leaves the chunk in eager form: dm = diag(sigma) dMh
        if (!fmask) {
#pragma unroll
            for (int r = 0; r < S; ++r) {
                const float f = s_fold[r];
#pragma unroll
                for (int cc = 0; cc < CPL; ++cc) dm[r][cc] *= f;
            }
        }
        __syncthreads();
        if (c >= 2) store_meta(c - 2, meta2);
        if (c >= 1) finish_stage(c - 1, sg);
    }
    // adjoint of the segment's initial state (FP32, per sequence)
    if (live) {
        const int64_t off = ((bidx * p.banks + bank) * p.heads + head) * S * p.width + col0;
#pragma unroll
        for (int r = 0; r < S; ++r)
            *reinterpret_cast<float2 *>(p.dinit + off + int64_t(r) * p.width) = make_float2(dm[r][0], dm[r][1]);
    }
}

// ------------------------------------------- other bank sizes and intervals

// Sums each of N values over the columns of a row group: the 64 / RG lanes of
// equal lane * RG / 64.  Value o ends in the lane of the group for which
// `at` = o and `mine` is set; other lanes return a partial sum.
template <int RG, int N>
__device__ __forceinline__ float reduce_columns(const float (&x)[N], int lane, int &at, bool &mine) {
    const int pos = lane & 15;
    if constexpr (RG == 1) {
        mine = pos < N / 4;
        at = (N / 4) * (lane >> 4) + (mine ? pos : 0);
        return reduce_scatter<N>(x, lane);
    } else {
        constexpr int M = RG == 2 ? N / 2 : N;
        mine = pos < M;
        at = (mine ? pos : 0) + (RG == 2 ? M * ((lane >> 4) & 1) : 0);
        float out = 0.f;
#pragma unroll
        for (int i = 0; i < M; ++i) {
            const float z = row_total(RG == 2 ? row_pair_sum(x[i], x[i + N - M]) : x[i]);
            out = pos == i ? z : out;
        }
        asm volatile("" : "+v"(out));  // computed in every lane, as in reduce_scatter
        return out;
    }
}

// Chunk replay for the shapes the S = 8 chunk kernel does not take: S in {4,
// 8, 16, 32} padded rows (s_real of them live), replay intervals C of 4, 8 or
// 16 events.  One workgroup of WAVES waves per (segment, head, tile of columns);
// chunks in reverse.  A lane owns CPL value columns and R = S / RG
// rows (at most 8): RG groups of 64 / RG lanes share a column's rows.
//  * All C states of a chunk sit in registers (C*R*CPL of them, at most 128),
//    so each write is replayed once.
//  * The operands of the next chunk (columns, row operands, start state) are
//    loaded when half of the chunk's events remain and put in LDS after them,
//    so no event waits for a load; the row operands (exp, bf(b p) k, bf(q r))
//    are formed once per event, spread over the lanes, not by every lane.
//  * The sums over columns (U, X, P, dq) are permlane swaps and DPP adds.  The
//    waves of a tile add theirs in LDS, so that a wave of 16 or 32 columns has
//    no rows of partial sums of its own in the workspace: with a row per wave it
//    was three times as large at S = 32, and the training step of 8,192 tokens,
//    H8 S16 v128, 256 banks took 3,148 us for 2,840, of 2,002 tokens, H4 S32
//    v64, 64 banks 635 for 544.
// Bound: instruction issue of the event loop.  Before it, one kernel loaded
// every operand at its event and reduced by shuffles: 813 -> 103 us at 16,384
// tokens, H1 S4 v128, 1024 banks (8,192 segments of 32 events), 1,934 -> 245
// us at 2,002 tokens, H4 S16 v64, 64 banks (128 segments of 250 events; 231
// with two one-wave workgroups in place of one of two, whose halves of the sums
// token_vjp_kernel read in 47 us for 38); of these, addresses and route slots by
// readlane took 115 -> 103 and 239 -> 229.  Two row groups at S = 16 (32 columns
// per wave) double the waves, which the second size needs to fill the chip, and
// halve a lane's states.
template <typename T, int S, int RG, int CPL, int C, int WAVES>
__global__ __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(2))) void staged_backward_kernel(
    BackwardParams<T> p) {
    constexpr int R = S / RG, kCols = kLanes / RG;
    constexpr bool kShared = WAVES > 1;
    constexpr int NR = (C * S + kLanes - 1) / kLanes;  // (event, row) operands per lane
    constexpr int kKey = 0, kDecay = S, kErase = 2 * S, kStride = 3 * S + 4;
    struct Staged {
        LaneCols<T, CPL> a[C], b[C];  // write: v, w; read: dy, dy
        T x[NR], bb[NR];             // write: k, b; read: q
        float g[NR];
        uint32_t m0[R][CPL];  // start state (BF16 or FP32 bits)
    };
    // each wave's own, but for the sums of a tile's waves by chunk % 3 (write: U, X, P; read: dq)
    __shared__ int4 s_meta_[WAVES][2][C];
    __shared__ __align__(16) float s_rows_[WAVES][C][kStride];
    __shared__ float s_cols_[WAVES][C][2 * CPL][kCols];  // write: v, bf(w p); read: dy
    __shared__ float s_part[kShared ? 3 : 1][WAVES][C][kShared ? 3 * S : 1];
    const int wave = kShared ? __builtin_amdgcn_readfirstlane(int(threadIdx.x) / kLanes) : 0;
    auto &s_meta = s_meta_[wave];
    auto &s_rows = s_rows_[wave];
    auto &s_cols = s_cols_[wave];

    int seg, head, tile;
    block_item(p, seg, head, tile);
    const int bank = seg % p.banks;
    const int64_t bidx = seg / p.banks;
    const int lane = kShared ? int(threadIdx.x) % kLanes : int(threadIdx.x);
    const int row0 = lane / kCols * R, col = lane % kCols;
    const int col0 = ((tile * WAVES + wave) * kCols + col) * CPL;
    const bool live = col0 < p.width;
    // waves of the tile with columns
    const int busy = min(WAVES, (p.width - tile * WAVES * kCols * CPL + kCols * CPL - 1) / (kCols * CPL));
    const int colc = live ? col0 : p.width - CPL;  // lanes past the width load valid columns and zero them
    const int64_t start = p.cu[seg], end = p.cu[seg + 1];
    const int count = int((end - start + C - 1) / C);
    const int64_t hw = int64_t(p.heads) * p.width;
    const int lane_col = head * p.width + colc;

    auto chunk_len = [&](int c) { return int(min(int64_t(C), end - (start + int64_t(c) * C))); };
    // Event lane % C of chunk c: token, route index within the token, is_read, route weight.
    auto load_meta = [&](int c) {
        const int64_t write_events = p.nt * p.kw, events = p.nt * (int64_t(p.kw) + p.kr);
        const int len = chunk_len(c);
        int64_t o = p.order[start + int64_t(c) * C + (lane < len ? lane : len - 1)];
        o = o < 0 ? 0 : (o >= events ? events - 1 : o);
        const bool rd = o >= write_events;
        const int64_t route = rd ? o - write_events : o;
        const int k = rd ? p.kr : p.kw;
        const int64_t token = p.k_shift >= 0 ? route >> p.k_shift
                                             : (events <= int64_t(UINT32_MAX) ? int64_t(uint32_t(route) / uint32_t(k)) : route / k);
        return make_int4(int(token), int(route - token * k), rd ? 1 : 0, __float_as_int(to_f32(rd ? p.rw[route] : p.ww[route])));
    };
    auto store_meta = [&](int c, const int4 &m) {
        if (lane < C) s_meta[c & 1][lane] = m;
    };
    // Loads of chunk c's operands and start state (its meta is in LDS); the
    // column addresses as in chunk_backward_kernel.
    auto issue_stage = [&](int c, Staged &sg) {
        const int len = chunk_len(c);
        const int4 *mt = s_meta[c & 1];
        const int ev = lane & (C - 1);
        const int4 me = mt[ev < len ? ev : len - 1];
        const int64_t row = int64_t(me.x) * hw;
        const uint64_t ra = reinterpret_cast<uint64_t>((me.z ? p.dy : p.v) + row);
        const uint64_t rb = reinterpret_cast<uint64_t>((me.z ? p.dy : p.w) + row);
        const uint32_t byte = uint32_t(lane_col) * uint32_t(sizeof(T));
#pragma unroll
        for (int e = 0; e < C; ++e) {
            sg.a[e].load(reinterpret_cast<const T *>(lane_ptr(ra, e) + byte));
            sg.b[e].load(reinterpret_cast<const T *>(lane_ptr(rb, e) + byte));
        }
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            const int idx = (lane + i * kLanes) & (C * S - 1), e = idx / S, r = idx % S;
            const int4 m = mt[e < len ? e : len - 1];
            const int64_t at = (int64_t(m.x) * p.heads + head) * p.s_real + (r < p.s_real ? r : 0);
            sg.x[i] = (m.z ? p.q : p.k)[at];
            sg.bb[i] = p.b[at];
            sg.g[i] = p.g[at];
        }
        const bool first = c == 0;
        const void *base = first ? p.initial : p.snap;
        const int64_t off = first ? bidx * p.init_bstride + (int64_t(bank) * p.heads + head) * p.s_real * p.width
                                  : (((start + int64_t(c) * C) / C - 1) * p.heads + head) * p.s_real * p.width;
        const bool half = (first ? p.init_dtype : p.snap_dtype) == BDM_BF16;
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int cc = 0; cc < CPL; ++cc) {
                const int64_t at = off + int64_t(row0 + r < p.s_real ? row0 + r : 0) * p.width + colc + cc;
                if (half) sg.m0[r][cc] = static_cast<const uint16_t *>(base)[at];
                else sg.m0[r][cc] = static_cast<const uint32_t *>(base)[at];
            }
    };
    // Operand rows and columns of chunk c into LDS, its start state into m0.
    auto finish_stage = [&](int c, const Staged &sg, float (&m0)[R][CPL]) {
        const int len = chunk_len(c);
        const int4 *mt = s_meta[c & 1];
        const int weight = mt[(lane & (C - 1)) < len ? lane & (C - 1) : len - 1].w;  // lane e: event e's
#pragma unroll
        for (int e = 0; e < C; ++e) {
            const float pw = __int_as_float(__builtin_amdgcn_readlane(weight, e));
#pragma unroll
            for (int cc = 0; cc < CPL; ++cc) {  // (the row groups of a column store the same values)
                s_cols[e][cc][col] = live ? sg.a[e].get(cc) : 0.f;
                s_cols[e][CPL + cc][col] = live ? round_to<T>(sg.b[e].get(cc) * pw) : 0.f;
            }
        }
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            const int idx = (lane + i * kLanes) & (C * S - 1), e = idx / S, r = idx % S;
            const int4 m = mt[e < len ? e : len - 1];
            const float pw = __int_as_float(m.w);
            const float x = r < p.s_real ? to_f32(sg.x[i]) : 0.f;
            if (m.z) {
                s_rows[e][kKey + r] = round_to<T>(x * pw) * p.scale;
            } else {  // prepare_write_rows of row r
                s_rows[e][kKey + r] = x;
                s_rows[e][kDecay + r] = r < p.s_real ? __expf(p.routed_decay ? sg.g[i] * pw : sg.g[i]) : 0.f;
                s_rows[e][kErase + r] = round_to<T>(to_f32(sg.bb[i]) * pw) * x;
            }
        }
        const bool half = (c == 0 ? p.init_dtype : p.snap_dtype) == BDM_BF16;
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int cc = 0; cc < CPL; ++cc) {
                float x = __uint_as_float(half ? sg.m0[r][cc] << 16 : sg.m0[r][cc]);
                if (c == 0 && p.rounding) x = round_bf16(x);
                m0[r][cc] = live && row0 + r < p.s_real ? x : 0.f;
            }
    };
    auto rows_of = [&](int e, int at, float (&x)[R]) {
        const float4 *row = reinterpret_cast<const float4 *>(&s_rows[e][at + row0]);
#pragma unroll
        for (int i = 0; i < R / 4; ++i) {
            const float4 f = row[i];
            x[4 * i] = f.x, x[4 * i + 1] = f.y, x[4 * i + 2] = f.z, x[4 * i + 3] = f.w;
        }
    };
    // One write on the state m before it (apply_write, its row sum over the row groups).
    auto apply = [&](int e, float (&m)[R][CPL]) {
        float kk[R], dd[R], a[R];
        rows_of(e, kKey, kk);
        rows_of(e, kDecay, dd);
        rows_of(e, kErase, a);
#pragma unroll
        for (int cc = 0; cc < CPL; ++cc) {
            float erase = 0.f;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                m[r][cc] *= dd[r];
                erase = fmaf(a[r], m[r][cc], erase);
            }
            const float u = fmaf(s_cols[e][CPL + cc][col], s_cols[e][cc][col], -sum_row_groups<RG>(erase));
#pragma unroll
            for (int r = 0; r < R; ++r) m[r][cc] = fmaf(kk[r], u, m[r][cc]);
        }
    };

    float dm[R][CPL];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int cc = 0; cc < CPL; ++cc) dm[r][cc] = 0.f;

    int sums = 0;  // the chunk's buffer of s_part
    // Route slot of event e from the chunk's metadata, lane e holding event e's.
    auto slot_of = [&](int e, const int4 &meta, int per_token) {
        return int64_t(__builtin_amdgcn_readlane(meta.x, e)) * per_token + __builtin_amdgcn_readlane(meta.y, e);
    };
    // Adjoint of write e with the state st before it.
    auto write_back = [&](int e, const int4 &meta, float (&st)[R][CPL]) {
        float kk[R], dd[R], a[R];
        rows_of(e, kKey, kk);
        rows_of(e, kDecay, dd);
        rows_of(e, kErase, a);
        float u[CPL], du[CPL];
#pragma unroll
        for (int cc = 0; cc < CPL; ++cc) {
            float erase = 0.f, acc = 0.f;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                st[r][cc] *= dd[r];  // hd
                erase = fmaf(a[r], st[r][cc], erase);
                acc = fmaf(dm[r][cc], kk[r], acc);
            }
            u[cc] = fmaf(s_cols[e][CPL + cc][col], s_cols[e][cc][col], -sum_row_groups<RG>(erase));
            du[cc] = sum_row_groups<RG>(acc);
        }
        const int64_t slot = slot_of(e, meta, p.kw);
        if (live && row0 == 0) {
            float *du_row = p.du + slot * hw + head * p.width + col0;
            if constexpr (CPL == 2) *reinterpret_cast<float2 *>(du_row) = make_float2(du[0], du[1]);
            else du_row[0] = du[0];
        }
        float *wp = p.wpart + ((int64_t(tile) * p.nt * p.kw + slot) * p.heads + head) * 3 * p.s_real;
#pragma unroll
        for (int g = 0; g < R / 4; ++g) {  // the group's rows 4g .. 4g + 3: red = U[4], X[4], P[4]
            float red[12];
#pragma unroll
            for (int i = 0; i < 12; ++i) red[i] = 0.f;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int r = 4 * g + i;
#pragma unroll
                for (int cc = 0; cc < CPL; ++cc) {
                    red[i] = fmaf(dm[r][cc], u[cc], red[i]);
                    red[4 + i] = fmaf(st[r][cc], du[cc], red[4 + i]);
                    red[8 + i] = fmaf(dm[r][cc], st[r][cc], red[8 + i]);
                    // dh <- (dh - a du^T) * decay (role_bank_kernel.py:130-138)
                    dm[r][cc] = (dm[r][cc] - a[r] * du[cc]) * dd[r];
                }
            }
            int at;
            bool mine;
            const float o = reduce_columns<RG, 12>(red, lane, at, mine);
            const int r = row0 + 4 * g + (at & 3);
            if constexpr (kShared) {
                if (mine) s_part[sums][wave][e][(at >> 2) * S + r] = o;
            } else {
                if (mine && r < p.s_real) wp[(at >> 2) * p.s_real + r] = o;
            }
        }
    };
    // Adjoint of read e with the state st it read: dq = scale st dy, dm += scale eq dy^T.
    auto read_back = [&](int e, const int4 &meta, const float (&st)[R][CPL]) {
        float eq[R], dy[CPL], red[R];
        rows_of(e, kKey, eq);
#pragma unroll
        for (int cc = 0; cc < CPL; ++cc) dy[cc] = s_cols[e][cc][col];
        float *rp = p.rpart + ((int64_t(tile) * p.nt * p.kr + slot_of(e, meta, p.kr)) * p.heads + head) * p.s_real;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            red[r] = 0.f;
#pragma unroll
            for (int cc = 0; cc < CPL; ++cc) {
                red[r] = fmaf(st[r][cc], dy[cc], red[r]);
                dm[r][cc] = fmaf(eq[r], dy[cc], dm[r][cc]);
            }
        }
        int at;
        bool mine;
        const float o = reduce_columns<RG, R>(red, lane, at, mine) * p.scale;
        if constexpr (kShared) {
            if (mine) s_part[sums][wave][e][row0 + at] = o;
        } else {
            if (mine && row0 + at < p.s_real) rp[row0 + at] = o;
        }
    };
    // The chunk's sums over the tile's waves, in wave order: wave w takes the events
    // w, w + WAVES, ..., a lane one or two of an event's 3S sums.  rows: lane e event
    // e's row of the workspace.
    auto store_sums = [&](int from, uint64_t rows, uint32_t wmask, uint32_t rmask) {
        constexpr int kEvents = C / WAVES, kPer = (3 * S + kLanes - 1) / kLanes;
        float sum[kEvents][kPer];
#pragma unroll
        for (int n = 0; n < kEvents; ++n)
#pragma unroll
            for (int q = 0; q < kPer; ++q) {
                const int i = min(lane + q * kLanes, 3 * S - 1);
                sum[n][q] = s_part[from][0][wave + n * WAVES][i];
#pragma unroll
                for (int w = 1; w < WAVES; ++w) sum[n][q] += w < busy ? s_part[from][w][wave + n * WAVES][i] : 0.f;
            }
#pragma unroll
        for (int n = 0; n < kEvents; ++n) {
            const int e = wave + n * WAVES;
            const int count = wmask >> e & 1u ? 3 * S : (rmask >> e & 1u ? S : 0);  // (a read has dq in U's place)
            float *row = reinterpret_cast<float *>(const_cast<char *>(lane_ptr(rows, e)));
#pragma unroll
            for (int q = 0; q < kPer; ++q) {
                const int i = lane + q * kLanes, r = i % S;
                if (i < count && r < p.s_real) row[i / S * p.s_real + r] = sum[n][q];
            }
        }
    };
    // (bases, strides and the difference in registers: a choice between two kernel arguments becomes a load of one)
    const int64_t wsums = (int64_t(tile) * p.nt * p.kw * p.heads + head) * 3 * p.s_real, wstride = int64_t(p.heads) * 3 * p.s_real;
    const int64_t rsums = (int64_t(tile) * p.nt * p.kr * p.heads + head) * p.s_real, rstride = int64_t(p.heads) * p.s_real;
    const uint64_t wbase = reinterpret_cast<uint64_t>(p.wpart + wsums), rbase = reinterpret_cast<uint64_t>(p.rpart + rsums);
    const int more = p.kr - p.kw;
    auto sums_row = [&](const int4 &meta) {
        const int64_t slot = int64_t(meta.x) * (p.kw + (meta.z ? more : 0)) + meta.y;
        return (meta.z ? rbase : wbase) + uint64_t(slot * (meta.z ? rstride : wstride)) * sizeof(float);
    };

    // The sums of the chunk before, stored once every wave of the tile has passed it: half a chunk later, so
    // that no wave waits for another's last event (a third buffer, since the others may be a chunk further).
    uint64_t done_rows = 0;
    uint32_t done_writes = 0, done_reads = 0;
    auto finish_sums = [&] {
        __syncthreads();
        store_sums(sums ? sums - 1 : 2, done_rows, done_writes, done_reads);
    };
    auto keep_sums = [&](const int4 &meta, uint32_t wmask, uint32_t rmask) {
        done_rows = sums_row(meta), done_writes = wmask, done_reads = rmask;
        sums = sums == 2 ? 0 : sums + 1;
    };
    if constexpr (kShared) {
        if (wave >= busy) {  // no columns: only its share of the sums
            for (int c = count - 1; c >= 0; --c) {
                const int4 mine = load_meta(c);
                const bool valid = lane < chunk_len(c);
                if (c < count - 1) finish_sums();
                keep_sums(mine, uint32_t(__ballot(valid && mine.z == 0)), uint32_t(__ballot(valid && mine.z != 0)));
            }
            if (count > 0) finish_sums();
            return;
        }
    }
    // Order among a wave's own LDS accesses (which run in order).
    auto sync_wave = [] {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    float m0[R][CPL];
    if (count > 0) {
        store_meta(count - 1, load_meta(count - 1));
        int4 prev = make_int4(0, 0, 0, 0);
        if (count > 1) prev = load_meta(count - 2);
        sync_wave();
        Staged sg;
        issue_stage(count - 1, sg);
        if (count > 1) store_meta(count - 2, prev);
        sync_wave();
        finish_stage(count - 1, sg, m0);
    }
#pragma unroll 1
    for (int c = count - 1; c >= 0; --c) {
        sync_wave();
        const int len = chunk_len(c);
        const int4 mine = s_meta[c & 1][lane & (C - 1)];
        const uint32_t wmask = uint32_t(__ballot(lane < len && mine.z == 0)) & ((1u << C) - 1);
        const uint32_t rmask = uint32_t(__ballot(lane < len && mine.z != 0)) & ((1u << C) - 1);
        float st[C][R][CPL];
#pragma unroll
        for (int e = 0; e < C; ++e) {
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int cc = 0; cc < CPL; ++cc) st[e][r][cc] = e ? st[e - 1][r][cc] : m0[r][cc];
            if (e && (wmask & (1u << (e - 1)))) apply(e - 1, st[e]);
        }
#pragma unroll
        for (int e = C - 1; e >= C / 2; --e) {
            if (wmask & (1u << e)) write_back(e, mine, st[e]);
            else if (rmask & (1u << e)) read_back(e, mine, st[e]);
        }
        // the next chunk's loads, in flight while the first half is differentiated
        int4 meta2 = make_int4(0, 0, 0, 0);
        Staged sg;
        if (c >= 2) meta2 = load_meta(c - 2);
        if (c >= 1) issue_stage(c - 1, sg);
        if (kShared && c < count - 1) finish_sums();
#pragma unroll
        for (int e = C / 2 - 1; e >= 0; --e) {
            if (wmask & (1u << e)) write_back(e, mine, st[e]);
            else if (rmask & (1u << e)) read_back(e, mine, st[e]);
        }
        sync_wave();
        if (c >= 2) store_meta(c - 2, meta2);
        if (c >= 1) finish_stage(c - 1, sg, m0);
        if constexpr (kShared) keep_sums(mine, wmask, rmask);
    }
    if (kShared && count > 0) finish_sums();
    // adjoint of the segment's initial state (FP32, per sequence)
    if (live) {
        const int64_t off = ((bidx * p.banks + bank) * p.heads + head) * p.s_real * p.width + col0;
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int cc = 0; cc < CPL; ++cc)
                if (row0 + r < p.s_real) p.dinit[off + int64_t(row0 + r) * p.width + cc] = dm[r][cc];
    }
}


template <typename T>
struct VjpParams {
    const T *q, *k, *b;
    const float *g;
    const T *v, *w;
    const T *ww, *rw;
    const float *du, *wpart, *rpart;
    T *dq, *dk, *db, *dv, *dw, *dww, *drw;
    float *dg;
    int64_t nt;
    int heads, s_real, width, kw, kr, tiles;
    int wph;  // token_grad_kernel: waves per head (each owns 64 * CPL value columns)
    int routed_decay;
};

__device__ __forceinline__ float wave_sum(float x) {
#pragma unroll
    for (int m = kLanes / 2; m >= 1; m >>= 1) x += __shfl_xor(x, m, kLanes);
    return x;
}

// Sum over the 8 lanes of an 8-lane group (lane % 8 varies), in every lane.
__device__ __forceinline__ float group8_sum(float x) {
    x += __shfl_xor(x, 1, kLanes);
    x += __shfl_xor(x, 2, kLanes);
    return x + __shfl_xor(x, 4, kLanes);
}

// Sum over the 8 lanes of equal lane % 8 (lane / 8 varies), in every lane.
__device__ __forceinline__ float stride8_sum(float x) {
    x += __shfl_xor(x, 8, kLanes);
    x += __shfl_xor(x, 16, kLanes);
    return x + __shfl_xor(x, 32, kLanes);
}

// One workgroup per token, one wave per head (heads <= 16); S <= 8, KW, KR
// <= 8 and width <= 64 * CPL * wph.  Bound: HBM, the FP32 du of a token's
// writes (537 MB at 8,192 tokens, 8 writes, 2,048 columns).  One load per
// slot and lane for its adjacent columns, and WAVES: a wide head's waves each
// load the tiles of their own columns for the S side instead of all of them:
// 311 -> 180 us there, 113 -> 86 at 8,192 tokens, H8 v128.  Lane (j, r) = (lane / 8, lane % 8) holds the
// S-side gradients of route slot j, row r; lane l owns value columns
// l*CPL .. l*CPL + CPL - 1.  The rounding points follow
// role_bank_dispatch.py:99-131; sums over slots and rows are in FP32.
template <typename T, int CPL, bool VEC, bool WAVES>
__global__ __launch_bounds__(1024) void token_grad_kernel(VjpParams<T> p) {
    constexpr int MAXH = 16, MAXK = 8, MAXW = 16;
    __shared__ float s_route[MAXH][2 * MAXK];  // per head: d(ww) of each write slot, then d(rw)
    __shared__ float s_wv[MAXW][MAXK];         // per wave: its columns' part of d(ww)
    const int64_t token = blockIdx.x;
    const int wave = threadIdx.x / kLanes, lane = threadIdx.x % kLanes;
    // a head's columns are split over p.wph waves; every wave of a head
    // computes the head's S-side terms, its first wave stores them
    const int head = wave / p.wph, hw = wave % p.wph;
    const int64_t row = token * p.heads + head;
    const int64_t wslots = p.nt * p.kw, rslots = p.nt * p.kr;
    const int j = lane >> 3, r = lane & 7;
    const bool srow = r < p.s_real;
    const bool wl = srow && j < p.kw, rl = srow && j < p.kr;
    const int64_t wslot = token * p.kw + (j < p.kw ? j : p.kw - 1);
    const int64_t rslot = token * p.kr + (j < p.kr ? j : p.kr - 1);
    const int rr = srow ? r : 0;

    // ---- every load first: the S side (slot j, row r), then the value columns
    const float q0 = to_f32(p.q[row * p.s_real + rr]);
    const float k0 = to_f32(p.k[row * p.s_real + rr]);
    const float b0 = to_f32(p.b[row * p.s_real + rr]);
    const float g0 = p.g[row * p.s_real + rr];
    const float pw = to_f32(p.ww[wslot]), pr = to_f32(p.rw[rslot]);
    // a wave's column tile of U, X, P and dq (a head of one wave sums its tiles itself)
    const auto tile_part = [&](int t, float (&x)[4]) {
        const float *wp = p.wpart + ((int64_t(t) * wslots + wslot) * p.heads + head) * 3 * p.s_real + rr;
        x[0] = wp[0], x[1] = wp[p.s_real], x[2] = wp[2 * p.s_real];
        x[3] = p.rpart[((int64_t(t) * rslots + rslot) * p.heads + head) * p.s_real + rr];
    };
    constexpr int kTilesPerWave = 2;  // of 128 columns, of a wave's 256 (WAVES)
    float part[kTilesPerWave][4];
    tile_part(WAVES ? min(hw * kTilesPerWave, p.tiles - 1) : 0, part[0]);
    if constexpr (WAVES) tile_part(min(hw * kTilesPerWave + 1, p.tiles - 1), part[1]);
    const int c0 = (hw * kLanes + lane) * CPL;
    bool live[CPL];
    float v0[CPL], w0[CPL], vwsum[CPL], wsum[CPL], wv[MAXK];
    // every slot's du and weight requested up front (slots >= KW re-read slot
    // KW-1: straight-line loads, all in flight together).  VEC: the width is a
    // multiple of CPL, so a lane's columns are one load and live together.
    float dus[MAXK][CPL], pws[MAXK];
    if constexpr (VEC) {
        const int cc = c0 < p.width ? c0 : p.width - CPL;  // lanes past the width re-read the last columns and drop them
        load_row<CPL>(p.v + row * p.width + cc, v0);
        load_row<CPL>(p.w + row * p.width + cc, w0);
#pragma unroll
        for (int jj = 0; jj < MAXK; ++jj) {
            const int64_t slot = token * p.kw + (jj < p.kw ? jj : p.kw - 1);
            pws[jj] = to_f32(p.ww[slot]);
            const float *du = p.du + (slot * p.heads + head) * p.width + cc;
            if constexpr (CPL == 2) {
                const float2 x = *reinterpret_cast<const float2 *>(du);
                dus[jj][0] = x.x, dus[jj][1] = x.y;
            } else {
                load_row<CPL>(du, dus[jj]);
            }
        }
    } else {
        int cols[CPL];  // clamped columns
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
            cols[c] = min(c0 + c, p.width - 1);
            v0[c] = to_f32(p.v[row * p.width + cols[c]]);
            w0[c] = to_f32(p.w[row * p.width + cols[c]]);
        }
#pragma unroll
        for (int jj = 0; jj < MAXK; ++jj) {
            const int64_t slot = token * p.kw + (jj < p.kw ? jj : p.kw - 1);
            pws[jj] = to_f32(p.ww[slot]);
            const float *du = p.du + (slot * p.heads + head) * p.width;
#pragma unroll
            for (int c = 0; c < CPL; ++c) dus[jj][c] = du[cols[c]];
        }
    }
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
        live[c] = c0 + c < p.width;
        v0[c] = live[c] ? v0[c] : 0.f;
        w0[c] = live[c] ? w0[c] : 0.f;
        vwsum[c] = wsum[c] = 0.f;
    }
    float su = part[0][0], sx = part[0][1], sp = part[0][2], sq = part[0][3];
    if constexpr (WAVES) {
        // each wave of a head loads its own tiles; the first adds them, in tile order
        __shared__ float s_part[MAXW * kTilesPerWave][4][kLanes];
#pragma unroll
        for (int n = 0; n < kTilesPerWave; ++n)
#pragma unroll
            for (int x = 0; x < 4; ++x) s_part[wave * kTilesPerWave + n][x][lane] = part[n][x];
        __syncthreads();
        if (hw == 0)
            for (int t = 1; t < p.tiles; ++t) {
                su += s_part[wave * kTilesPerWave + t][0][lane];
                sx += s_part[wave * kTilesPerWave + t][1][lane];
                sp += s_part[wave * kTilesPerWave + t][2][lane];
                sq += s_part[wave * kTilesPerWave + t][3][lane];
            }
    } else {
        for (int t = 1; t < p.tiles; ++t) {  // column tiles past the first
            tile_part(t, part[1]);
            su += part[1][0];
            sx += part[1][1];
            sp += part[1][2];
            sq += part[1][3];
        }
    }
    float wb = 0.f, wr = 0.f, dec = 0.f;
    if (!WAVES || hw == 0) {
        // dk = U - eb X ; db = -k X ; dg = P - a X (role_bank_kernel.py:128-135)
        const float eb = round_to<T>(b0 * pw);
        const float dk = round_to<T>(su - eb * sx);
        const float db = round_to<T>(-k0 * sx);
        const float dg = sp - eb * k0 * sx;
        // routed decay: the packed gate was g*p (routed_update.py:43-47)
        const float k_term = wl ? dk : 0.f;
        const float g_term = wl ? (p.routed_decay ? dg * pw : dg) : 0.f;
        const float b_term = wl ? round_to<T>(db * pw) : 0.f;
        wb = round_to<T>(group8_sum(wl ? round_to<T>(db * b0) : 0.f));
        dec = group8_sum(wl ? dg * g0 : 0.f);
        const float dq = round_to<T>(sq);
        const float q_term = rl ? round_to<T>(dq * pr) : 0.f;
        wr = round_to<T>(group8_sum(rl ? round_to<T>(dq * q0) : 0.f));
        const float kwsum = stride8_sum(k_term), gsum = stride8_sum(g_term), bsum = stride8_sum(b_term);
        const float qsum = stride8_sum(q_term);
        if (j == 0 && srow) {
            const int64_t at = row * p.s_real + r;
            p.dq[at] = from_f32<T>(qsum);
            p.dk[at] = from_f32<T>(kwsum);
            p.dg[at] = gsum;
            p.db[at] = from_f32<T>(bsum);
        }
    }

    // ---- value columns: the token's write events in route order
#pragma unroll
    for (int jj = 0; jj < MAXK; ++jj) {
        wv[jj] = 0.f;
        if (jj < p.kw) {
            const float pj = pws[jj];
#pragma unroll
            for (int c = 0; c < CPL; ++c) {
                const float d = live[c] ? dus[jj][c] : 0.f;
                const float ew = round_to<T>(w0[c] * pj);
                const float dv = round_to<T>(d * ew);
                const float dw = round_to<T>(d * v0[c]);
                vwsum[c] = round_to<T>(vwsum[c] + dv);
                wsum[c] = round_to<T>(wsum[c] + round_to<T>(dw * pj));
                wv[jj] += round_to<T>(dw * w0[c]);
            }
        }
    }
    if constexpr (VEC) {
        if (live[0]) {
            if constexpr (CPL == 2) {
                store_cols(p.dv + row * p.width + c0, vwsum);
                store_cols(p.dw + row * p.width + c0, wsum);
            } else {
                store_row<CPL>(p.dv + row * p.width + c0, vwsum);
                store_row<CPL>(p.dw + row * p.width + c0, wsum);
            }
        }
    } else {
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
            if (live[c]) {
                p.dv[row * p.width + c0 + c] = from_f32<T>(vwsum[c]);
                p.dw[row * p.width + c0 + c] = from_f32<T>(wsum[c]);
            }
        }
    }
    const float wv_total = reduce_scatter<MAXK>(wv, lane);
    if ((lane & 15) < MAXK / 4) s_wv[wave][(MAXK / 4) * (lane >> 4) + (lane & 15)] = wv_total;
    __syncthreads();
    if (hw == 0 && r == 0) {
        if (j < p.kw) {
            float cols = 0.f;  // the head's waves in column order
            for (int w = 0; w < p.wph; ++w) cols += s_wv[wave + w][j];
            float dww = round_to<T>(wb + round_to<T>(cols));
            if (p.routed_decay) dww = round_to<T>(dww + dec);
            s_route[head][j] = dww;
        }
        if (j < p.kr) s_route[head][MAXK + j] = wr;
    }
    __syncthreads();
    // route-weight gradients: the heads' contributions added in head order
    if (threadIdx.x < unsigned(p.kw + p.kr)) {
        const int jj = threadIdx.x;
        const bool wr_ = jj < p.kw;
        const int col = wr_ ? jj : MAXK + jj - p.kw;
        float total = 0.f;
        for (int h = 0; h < p.heads; ++h) total += s_route[h][col];
        if (wr_) p.dww[token * p.kw + jj] = from_f32<T>(total);
        else p.drw[token * p.kr + (jj - p.kw)] = from_f32<T>(total);
    }
}


// One workgroup (4 waves) per token.  VPL = value columns per lane.
template <typename T, int VPL>
__global__ __launch_bounds__(256) void token_vjp_kernel(VjpParams<T> p) {
    extern __shared__ float s_route[];  // [H][KW] d(ww) then [H][KR] d(rw), per head
    const int64_t token = blockIdx.x;
    const int wave = threadIdx.x / kLanes, lane = threadIdx.x % kLanes;
    const int nwaves = blockDim.x / kLanes;
    const int64_t wslots = p.nt * p.kw, rslots = p.nt * p.kr;
    const int64_t hs = int64_t(p.heads) * p.s_real;
    for (int head = wave; head < p.heads; head += nwaves) {
        const int64_t row = token * p.heads + head;
        const bool srow = lane < p.s_real;
        const float q0 = srow ? to_f32(p.q[row * p.s_real + lane]) : 0.f;
        const float k0 = srow ? to_f32(p.k[row * p.s_real + lane]) : 0.f;
        const float b0 = srow ? to_f32(p.b[row * p.s_real + lane]) : 0.f;
        const float g0 = srow ? p.g[row * p.s_real + lane] : 0.f;
        float v0[VPL], w0[VPL], vwsum[VPL], wsum[VPL];
#pragma unroll
        for (int i = 0; i < VPL; ++i) {
            const int c = lane + i * kLanes;
            v0[i] = c < p.width ? to_f32(p.v[row * p.width + c]) : 0.f;
            w0[i] = c < p.width ? to_f32(p.w[row * p.width + c]) : 0.f;
            vwsum[i] = wsum[i] = 0.f;
        }
        float kwsum = 0.f, gsum = 0.f, bsum = 0.f, qsum = 0.f;
        // write events in route order (role_bank_dispatch.py:99-115)
        for (int j = 0; j < p.kw; ++j) {
            const int64_t slot = token * p.kw + j;
            const float pw = to_f32(p.ww[slot]);
            float wb_part = 0.f, dec_part = 0.f;
            if (srow) {
                float su = 0.f, sx = 0.f, sp = 0.f;
                for (int t = 0; t < p.tiles; ++t) {
                    const float *wp = p.wpart + ((int64_t(t) * wslots + slot) * p.heads + head) * 3 * p.s_real;
                    su += wp[lane];
                    sx += wp[p.s_real + lane];
                    sp += wp[2 * p.s_real + lane];
                }
                // dk = U - eb X ; db = -k X ; dg = P - a X (role_bank_kernel.py:128-135)
                const float eb = round_to<T>(b0 * pw);
                const float dk = round_to<T>(su - eb * sx);
                const float db = round_to<T>(-k0 * sx);
                const float dg = sp - eb * k0 * sx;
                kwsum += dk;
                // routed decay: the packed gate was g*p (routed_update.py:43-47)
                gsum += p.routed_decay ? dg * pw : dg;
                dec_part = dg * g0;
                bsum += round_to<T>(db * pw);
                wb_part = round_to<T>(db * b0);
            }
            float wv_part = 0.f;
            const float *du = p.du + (slot * p.heads + head) * p.width;
#pragma unroll
            for (int i = 0; i < VPL; ++i) {
                const int c = lane + i * kLanes;
                if (c < p.width) {
                    const float ew = round_to<T>(w0[i] * pw);
                    const float dv = round_to<T>(du[c] * ew);
                    const float dw = round_to<T>(du[c] * v0[i]);
                    vwsum[i] = round_to<T>(vwsum[i] + dv);
                    wsum[i] = round_to<T>(wsum[i] + round_to<T>(dw * pw));
                    wv_part += round_to<T>(dw * w0[i]);
                }
            }
            const float wb = round_to<T>(wave_sum(wb_part));
            const float wv = round_to<T>(wave_sum(wv_part));
            float dww = round_to<T>(wb + wv);
            if (p.routed_decay) dww = round_to<T>(dww + wave_sum(dec_part));
            if (lane == 0) s_route[head * p.kw + j] = dww;
        }
        // read events in route order (:116-125)
        for (int j = 0; j < p.kr; ++j) {
            const int64_t slot = token * p.kr + j;
            const float pr = to_f32(p.rw[slot]);
            float wr_part = 0.f;
            if (srow) {
                float dq = 0.f;
                for (int t = 0; t < p.tiles; ++t) dq += p.rpart[(int64_t(t) * rslots + slot) * hs + head * p.s_real + lane];
                dq = round_to<T>(dq);
                qsum += round_to<T>(dq * pr);
                wr_part = round_to<T>(dq * q0);
            }
            const float wr = round_to<T>(wave_sum(wr_part));
            if (lane == 0) s_route[p.heads * p.kw + head * p.kr + j] = wr;
        }
        if (srow) {
            const int64_t at = row * p.s_real + lane;
            p.dq[at] = from_f32<T>(qsum);
            p.dk[at] = from_f32<T>(kwsum);
            p.dg[at] = gsum;
            p.db[at] = from_f32<T>(bsum);
        }
#pragma unroll
        for (int i = 0; i < VPL; ++i) {
            const int c = lane + i * kLanes;
            if (c < p.width) {
                p.dv[row * p.width + c] = from_f32<T>(vwsum[i]);
                p.dw[row * p.width + c] = from_f32<T>(wsum[i]);
            }
        }
    }
    __syncthreads();
    // route-weight gradients: the heads' contributions added in head order
    for (int j = threadIdx.x; j < p.kw + p.kr; j += blockDim.x) {
        float total = 0.f;
        if (j < p.kw) {
            for (int h = 0; h < p.heads; ++h) total += s_route[h * p.kw + j];
            p.dww[token * p.kw + j] = from_f32<T>(total);
        } else {
            const int jr = j - p.kw;
            for (int h = 0; h < p.heads; ++h) total += s_route[p.heads * p.kw + h * p.kr + jr];
            p.drw[token * p.kr + jr] = from_f32<T>(total);
        }
    }
}

struct Workspace {
    float *du, *wpart, *rpart;
    int4 *meta;      // per-event meta of the S = 8 chunk kernel (null otherwise)
    int *seg_order;  // longest-first segment order (null: bank order)
    size_t bytes;
};

constexpr size_t align256(size_t x) { return (x + 255) / 256 * 256; }

int replay_interval(const bdm_backward_args &a) {
    return a.round_interval > 0 ? a.round_interval : a.snapshot_interval;
}

// The S = 8, interval-16 chunk kernel: even head width (column pairs) and
// token and route indices in 32 bits.
bool chunk_path(const bdm_backward_args &a) {
    const int64_t nt = a.batch * a.time;
    const int64_t k = a.write_banks > a.read_banks ? a.write_banks : a.read_banks;
    return a.bank_size == 8 && replay_interval(a) == 16 && a.head_width % 2 == 0 && a.write_banks >= 1 &&
           a.read_banks >= 1 && nt * k < INT32_MAX;
}

// Row groups of the staged kernel: at most 8 rows per lane.
int row_groups(const bdm_backward_args &a) { return a.bank_size <= 8 ? 1 : (a.bank_size <= 16 ? 2 : 4); }

// Value columns of a lane: pairs in the chunk kernel and, in the staged one,
// for banks of up to 4 rows whose heads fill more than 64 lanes (16 states of
// 4 x 2 values then take the registers that 8 x 1 values of larger banks
// take); loads of a pair need an even width.
int columns_per_lane(const bdm_backward_args &a) {
    if (chunk_path(a)) return 2;
    return a.bank_size <= 4 && a.head_width % 2 == 0 && a.head_width > kLanes ? 2 : 1;
}

// Columns of a tile, the unit of the partial sums over columns in the
// workspace, and the waves of a workgroup that share it.
int tile_columns(const bdm_backward_args &a) { return a.bank_size <= 8 ? 2 * kLanes : kLanes; }

int column_tiles(const bdm_backward_args &a) { return (a.head_width + tile_columns(a) - 1) / tile_columns(a); }

int tile_waves(const bdm_backward_args &a) {
    const int columns = kLanes / (chunk_path(a) ? 1 : row_groups(a)) * columns_per_lane(a);
    const int waves = std::min(tile_columns(a) / columns, (a.head_width + columns - 1) / columns);
    return waves == 3 ? 4 : waves;
}

// The per-token gradient kernel: one wave per head and one lane per (slot, row).
// A head wider than 256 columns takes ceil(width / 256) waves (4 columns per
// lane); the workgroup holds at most 16 waves.
int token_grad_waves(const bdm_backward_args &a) {
    return a.head_width <= 256 ? 1 : (a.head_width + 255) / 256;
}

bool token_grad_path(const bdm_backward_args &a) {
    return a.bank_size <= 8 && a.write_banks >= 1 && a.write_banks <= 8 && a.read_banks >= 1 && a.read_banks <= 8 &&
           a.heads * token_grad_waves(a) <= 16;
}

Workspace carve(const bdm_backward_args &a, void *base) {
    const size_t nt = size_t(a.batch) * size_t(a.time);
    const size_t hs = size_t(a.heads) * size_t(a.bank_size);
    const size_t tiles = size_t(column_tiles(a));
    const size_t du = align256(nt * a.write_banks * a.heads * size_t(a.head_width) * sizeof(float));
    const size_t wp = align256(tiles * 3 * nt * a.write_banks * hs * sizeof(float));
    const size_t rp = align256(tiles * nt * a.read_banks * hs * sizeof(float));
    const size_t mt = chunk_path(a) ? align256(nt * size_t(a.write_banks + a.read_banks) * sizeof(int4)) : 0;
    const int64_t nseg = int64_t(a.batch) * a.bank_count;
    const size_t so = order_geometry(nseg) ? align256(size_t(nseg) * sizeof(int)) : 0;
    char *c = static_cast<char *>(base);
    Workspace w{};
    w.du = reinterpret_cast<float *>(c);
    w.wpart = reinterpret_cast<float *>(c ? c + du : nullptr);
    w.rpart = reinterpret_cast<float *>(c ? c + du + wp : nullptr);
    w.meta = reinterpret_cast<int4 *>(c && mt ? c + du + wp + rp : nullptr);
    w.seg_order = reinterpret_cast<int *>(c && so && order_enabled() ? c + du + wp + rp + mt : nullptr);
    w.bytes = du + wp + rp + mt + so;
    return w;
}

template <typename T, bool CHUNK>
int launch_backward(const bdm_backward_args &a, const Workspace &ws, void (*kernel)(BackwardParams<T>),
                    hipStream_t stream) {
    BackwardParams<T> p{};
    p.q = static_cast<const T *>(a.q);
    p.k = static_cast<const T *>(a.k);
    p.b = static_cast<const T *>(a.b);
    p.g = a.g;
    p.v = static_cast<const T *>(a.v);
    p.w = static_cast<const T *>(a.w);
    p.ww = static_cast<const T *>(a.write_weights);
    p.rw = static_cast<const T *>(a.read_weights);
    p.order = a.order;
    p.cu = a.cu_seqlens;
    p.initial = a.initial;
    p.snap = a.snapshots;
    p.dy = static_cast<const T *>(a.grad_output);
    p.du = ws.du;
    p.wpart = ws.wpart;
    p.rpart = ws.rpart;
    p.dinit = a.grad_initial;
    p.init_bstride = a.initial_batch_stride;
    p.nt = a.batch * a.time;
    p.heads = a.heads;
    p.s_real = a.bank_size;
    p.width = a.head_width;
    p.banks = a.bank_count;
    p.kw = a.write_banks;
    p.kr = a.read_banks;
    p.tiles = column_tiles(a);
    p.k_shift = -1;
    for (int sh = 0; sh < 8; ++sh)
        if (a.write_banks == (1 << sh) && a.read_banks == (1 << sh)) p.k_shift = sh;
    p.init_dtype = a.initial_dtype;
    p.snap_dtype = a.snapshot_dtype;
    p.routed_decay = a.routed_decay;
    p.rounding = a.round_interval > 0;
    p.scale = a.scale;
    const int64_t nseg = a.batch * a.bank_count;
    p.xcd_remap = (nseg % 8 == 0) ? 1 : 0;
    const dim3 grid(unsigned(nseg), unsigned(a.heads), unsigned(p.tiles));
    const int threads = tile_waves(a) * kLanes;
    if constexpr (CHUNK) {
        const int64_t events = p.nt * (p.kw + p.kr);
        const unsigned blocks = unsigned((events + 255) / 256);
        event_meta_kernel<T><<<blocks, 256, 0, stream>>>(p.order, events, p.nt * p.kw, p.kw, p.kr, p.ww, p.rw, ws.meta);
        if (int rc = check_launch("event_meta_kernel")) return rc;
        p.meta = ws.meta;
    }
    if (ws.seg_order) {
        launch_segment_order(p.cu, nseg, ws.seg_order, stream);
        if (int rc = check_launch("segment_order_kernel")) return rc;
        p.seg_order = ws.seg_order;
        p.order_gpr = order_groups_per_round(reinterpret_cast<const void *>(kernel), threads, nseg,
                                             int(grid.y * grid.z));
    }
    kernel<<<grid, threads, 0, stream>>>(p);
    if (int rc = check_launch(CHUNK ? "chunk_backward_kernel" : "staged_backward_kernel")) return rc;

    VjpParams<T> v{};
    v.q = p.q;
    v.k = p.k;
    v.b = p.b;
    v.g = p.g;
    v.v = p.v;
    v.w = p.w;
    v.ww = p.ww;
    v.rw = p.rw;
    v.du = ws.du;
    v.wpart = ws.wpart;
    v.rpart = ws.rpart;
    v.dq = static_cast<T *>(a.grad_q);
    v.dk = static_cast<T *>(a.grad_k);
    v.db = static_cast<T *>(a.grad_b);
    v.dv = static_cast<T *>(a.grad_v);
    v.dw = static_cast<T *>(a.grad_w);
    v.dww = static_cast<T *>(a.grad_write_weights);
    v.drw = static_cast<T *>(a.grad_read_weights);
    v.dg = a.grad_g;
    v.nt = p.nt;
    v.heads = a.heads;
    v.s_real = a.bank_size;
    v.width = a.head_width;
    v.kw = a.write_banks;
    v.kr = a.read_banks;
    v.tiles = p.tiles;
    v.routed_decay = a.routed_decay;
    v.wph = token_grad_waves(a);
    const unsigned blocks = unsigned(p.nt);
    if (token_grad_path(a)) {
        const unsigned threads = unsigned(a.heads * v.wph) * kLanes;
        auto launch = [&](auto cpl, auto waves) {
            constexpr int CPL = decltype(cpl)::value;
            constexpr bool WAVES = decltype(waves)::value;
            // (one column a lane is one load either way)
            if (CPL > 1 && a.head_width % CPL == 0)
                token_grad_kernel<T, CPL, (CPL > 1), WAVES><<<blocks, threads, 0, stream>>>(v);
            else
                token_grad_kernel<T, CPL, false, WAVES><<<blocks, threads, 0, stream>>>(v);
        };
        constexpr std::integral_constant<int, 4> four{};
        // the head's waves share its tiles of 128 columns (tile_columns up to 8 rows)
        if (v.wph > 1 && p.tiles <= 2 * v.wph)
            launch(four, std::true_type{});
        else if (v.wph > 1 || a.head_width > 2 * kLanes)
            launch(four, std::false_type{});
        else if (a.head_width > kLanes)
            launch(std::integral_constant<int, 2>{}, std::false_type{});
        else
            launch(std::integral_constant<int, 1>{}, std::false_type{});
        return check_launch("token_grad_kernel");
    }
    const size_t lds = size_t(a.heads) * size_t(a.write_banks + a.read_banks) * sizeof(float);
    if (a.head_width <= kLanes)
        token_vjp_kernel<T, 1><<<blocks, 256, lds, stream>>>(v);
    else if (a.head_width <= 2 * kLanes)
        token_vjp_kernel<T, 2><<<blocks, 256, lds, stream>>>(v);
    else if (a.head_width <= 4 * kLanes)
        token_vjp_kernel<T, 4><<<blocks, 256, lds, stream>>>(v);
    else if (a.head_width <= 8 * kLanes)
        token_vjp_kernel<T, 8><<<blocks, 256, lds, stream>>>(v);
    else if (a.head_width <= 16 * kLanes)
        token_vjp_kernel<T, 16><<<blocks, 256, lds, stream>>>(v);
    else
        token_vjp_kernel<T, 32><<<blocks, 256, lds, stream>>>(v);
    return check_launch("token_vjp_kernel");
}

template <typename T, int S, int C>
int launch_staged(const bdm_backward_args &a, const Workspace &ws, hipStream_t stream) {
    constexpr int RG = S <= 8 ? 1 : S / 8;  // row_groups
    auto launch = [&](auto cpl, auto waves) {
        return launch_backward<T, false>(
            a, ws, &staged_backward_kernel<T, S, RG, decltype(cpl)::value, C, decltype(waves)::value>, stream);
    };
    constexpr std::integral_constant<int, 1> one{};
    constexpr std::integral_constant<int, 2> two{};
    if constexpr (S == 4) {
        if (columns_per_lane(a) == 2) return launch(two, one);
    }
    if constexpr (S == 32) {
        if (tile_waves(a) == 4) return launch(one, std::integral_constant<int, 4>{});
    }
    return tile_waves(a) == 2 ? launch(one, two) : launch(one, one);
}

template <typename T>
int dispatch_backward(const bdm_backward_args &a, const Workspace &ws, hipStream_t stream) {
    const int c = replay_interval(a);
    if (chunk_path(a))
        return launch_backward<T, true>(a, ws,
                                        a.snapshot_dtype == BDM_BF16 ? &chunk_backward_kernel<T, bf16_t>
                                                                     : &chunk_backward_kernel<T, float>,
                                        stream);
    if (a.bank_size <= 4) {
        if (c == 16) return launch_staged<T, 4, 16>(a, ws, stream);
        if (c == 8) return launch_staged<T, 4, 8>(a, ws, stream);
        if (c == 4) return launch_staged<T, 4, 4>(a, ws, stream);
    } else if (a.bank_size <= 8) {
        if (c == 16) return launch_staged<T, 8, 16>(a, ws, stream);
        if (c == 8) return launch_staged<T, 8, 8>(a, ws, stream);
        if (c == 4) return launch_staged<T, 8, 4>(a, ws, stream);
    } else if (a.bank_size <= 16) {
        if (c == 8) return launch_staged<T, 16, 8>(a, ws, stream);
        if (c == 4) return launch_staged<T, 16, 4>(a, ws, stream);
    } else if (a.bank_size <= 32) {
        if (c == 4) return launch_staged<T, 32, 4>(a, ws, stream);
    }
    return fail(BDM_ERR_UNSUPPORTED, "backward: bank_size %d with replay interval %d", a.bank_size, c);
}

}  // namespace
}  // namespace bdm

extern "C" size_t bdm_backward_workspace_size(const bdm_backward_args *a) {
    if (!a || a->batch <= 0 || a->time <= 0 || a->heads <= 0 || a->head_width <= 0 || a->bank_size <= 0 ||
        a->write_banks < 0 || a->read_banks < 0)
        return 0;
    return bdm::carve(*a, nullptr).bytes;
}

extern "C" int bdm_backward(const bdm_backward_args *a, void *workspace, size_t workspace_bytes, void *stream) {
    using namespace bdm;
    if (!a) return fail(BDM_ERR_INVALID, "backward: null args");
    if (a->batch <= 0 || a->time <= 0 || a->heads <= 0 || a->bank_size <= 0 || a->head_width <= 0 ||
        a->bank_count <= 0 || a->write_banks < 0 || a->read_banks < 0 || a->write_banks + a->read_banks == 0)
        return fail(BDM_ERR_INVALID, "backward: bad geometry");
    if (a->head_width > 32 * kLanes) return fail(BDM_ERR_UNSUPPORTED, "backward: head_width %d > 2048", a->head_width);
    if (a->ctrl_dtype != BDM_BF16 && a->ctrl_dtype != BDM_F32)
        return fail(BDM_ERR_INVALID, "backward: ctrl dtype %d", a->ctrl_dtype);
    if ((a->initial_dtype != BDM_BF16 && a->initial_dtype != BDM_F32) ||
        (a->snapshot_dtype != BDM_BF16 && a->snapshot_dtype != BDM_F32))
        return fail(BDM_ERR_INVALID, "backward: state dtype");
    if (a->round_interval > 0 && a->snapshot_interval != a->round_interval)
        return fail(BDM_ERR_INVALID, "backward: snapshot interval must equal the rounding interval");
    if (a->round_interval == 0 && a->snapshot_dtype != BDM_F32)
        return fail(BDM_ERR_INVALID, "backward: an unrounded state needs FP32 snapshots");
    if (a->batch * a->bank_count > int64_t(INT32_MAX) || a->heads > 65535 ||
        a->batch * a->time > int64_t(INT32_MAX))
        return fail(BDM_ERR_UNSUPPORTED, "backward: grid too large");
    if (!a->q || !a->k || !a->g || !a->b || !a->v || !a->w || !a->write_weights || !a->read_weights ||
        !a->order || !a->cu_seqlens || !a->initial || !a->snapshots || !a->grad_output || !a->grad_q ||
        !a->grad_k || !a->grad_g || !a->grad_b || !a->grad_v || !a->grad_w || !a->grad_write_weights ||
        !a->grad_read_weights || !a->grad_initial)
        return fail(BDM_ERR_INVALID, "backward: null pointer");
    const Workspace need = carve(*a, nullptr);
    if (!workspace || workspace_bytes < need.bytes)
        return fail(BDM_ERR_WORKSPACE, "backward: workspace %zu < %zu bytes", workspace_bytes, need.bytes);
    if (!aligned(workspace, 256)) return fail(BDM_ERR_INVALID, "backward: workspace must be 256-byte aligned");
    const Workspace ws = carve(*a, workspace);
    hipStream_t s = as_stream(stream);
    if (a->ctrl_dtype == BDM_BF16) return dispatch_backward<bf16_t>(*a, ws, s);
    return dispatch_backward<float>(*a, ws, s);
}

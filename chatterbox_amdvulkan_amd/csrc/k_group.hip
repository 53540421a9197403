// k_group.hip -- a node list's small launches, several per kernel.
//
// A flow step's or a token's node list holds tens of launches that each move
// a few KB to a few MB: what bounds them is the launch (2.2 us from one
// kernel of a replayed graph to the next, 4 to 5 with several MB of dirty
// cache lines between), not the work.  Two forms, both bit-identical to the
// launches they replace (the same f32 operations in the same order per
// element, the LayerNorm reductions of k_ln_ext):
//
//   k_elt_group   independent element-wise ops side by side, one float4 a
//                 lane, a range of workgroups each
//   k_row_chain   dependent row ops (residual joins, LayerNorms, masks) on
//                 the same rows one after another: every op reads the row of
//                 the one before it, so the row stays in the registers of the
//                 waves that own it and no grid-wide order is needed.  What
//                 bounds a link is its two f64 reductions and its divisions
//                 (about 0.9 us with one row of 1024); its operands do not
//                 depend on the chain and are loaded three links ahead (one
//                 ahead: 1.5 us a link), its arguments a dozen links at once.
//
// Both are taken only where the launches are bound by their start (the
// schedule's limits, in floats and rows a CU): past them the one float4 a
// lane and the one row a workgroup lose to the launches' own kernels.
//
// Measured (a replay, us, before -> with both forms): a T3 token's 121
// launches 240 -> 61, the flow decoder's 80 on 500 frames 293 -> 187, the
// flow encoder's 48 on 125 tokens 129 -> 55.  These lists hold every matmul's
// output; between two matmuls of a running graph stand one to three
// launches: LayerNorm -> Mish -> mask -> + time embedding on 500 x 256, with a
// copy after it, 7.8 -> 6.7, bias + LayerNorm -> scale on 125 x 512 7.3 -> 6.4.
#include "cbx_rowops.h"

namespace cbx {
namespace {

constexpr int kThreads = 256;

struct EltArgs {
    int32_t n;
    uint32_t first[kEltMax];    // first workgroup of each op
    const uint16_t* tab;
    EltOp op[kEltMax];
};
static_assert(sizeof(EltArgs) <= 4096, "element-wise group arguments must fit the kernel argument segment");

__device__ __forceinline__ float4 elt_operand(const float* b, int mode, uint32_t i, uint32_t C, uint32_t ne0_4) {
    if (mode == kEltVec) return *reinterpret_cast<const float4*>(b + (4u * i) % C);
    if (mode == kEltFull) return *reinterpret_cast<const float4*>(b + 4ull * i);
    if (mode == kEltRowAny) {
        const uint32_t e = 4u * i;
        return make_float4(b[(e / ne0_4) % C], b[((e + 1) / ne0_4) % C], b[((e + 2) / ne0_4) % C], b[((e + 3) / ne0_4) % C]);
    }
    const float s = b[(i / ne0_4) % C];   // kEltRow
    return make_float4(s, s, s, s);
}

__global__ __launch_bounds__(kThreads) void k_elt_group(EltArgs a) {
    // offsets past the last op are ones no workgroup reaches: all of them
    // arrive in one batch of argument loads
    int k = 0;
#pragma unroll
    for (int j = 1; j < kEltMax; j++) k += blockIdx.x >= a.first[j] ? 1 : 0;
    const EltOp op = a.op[k];
    const uint32_t i = (blockIdx.x - a.first[k]) * kThreads + threadIdx.x;
    if (i >= op.n4) return;
    float4 v[1] = {Stream<float>::load4(reinterpret_cast<const char*>(op.x + 4ull * i))};
    if (op.bmode != kEltNone) {
        const float4 b = elt_operand(op.b, op.bmode, i, op.C, op.ne0_4);
        if (op.mul) v[0] = make_float4(v[0].x * b.x, v[0].y * b.y, v[0].z * b.z, v[0].w * b.w);
        else v[0] = make_float4(v[0].x + b.x, v[0].y + b.y, v[0].z + b.z, v[0].w + b.w);
    }
    if (op.b2) {
        const float4 b = *reinterpret_cast<const float4*>(op.b2 + (4u * i) % op.C2);
        v[0] = make_float4(v[0].x + b.x, v[0].y + b.y, v[0].z + b.z, v[0].w + b.w);
    }
    if (op.act == kEltScale) v[0] = make_float4(v[0].x * op.param, v[0].y * op.param, v[0].z * op.param, v[0].w * op.param);
    else if (op.act != CBX_UNARY_NONE) apply_act_vec<1>(op.act, v, a.tab, op.param);
    uint64_t o = i;
    if (op.ld4) {
        const uint32_t row = i / op.ne0_4;
        o = static_cast<uint64_t>(row) * op.ld4 + (i - row * op.ne0_4);
    }
    Stream<float>::store4(reinterpret_cast<char*>(op.y + 4 * o), v[0]);
}

// ---- row chain ------------------------------------------------------------------

struct ChainArgs {
    int32_t n, ne0;
    const uint16_t* tab;
    RowLink l[kChainMax];
};
static_assert(sizeof(ChainArgs) <= 4096, "row chain arguments must fit the kernel argument segment");

// One row a workgroup of WPR waves, NV float4s a lane (wave w holds float4s
// [w*64*NV, (w+1)*64*NV) of the row).
template <int NV, int WPR>
__global__ __launch_bounds__(64 * WPR) void k_row_chain(ChainArgs p) {
    __shared__ double lds[2 * WPR];
    const int lane = (threadIdx.x >> 6) * 64 * NV + (threadIdx.x & 63);
    const uint32_t row = blockIdx.x;
    const int64_t ne0 = p.ne0, ro = static_cast<int64_t>(row) * ne0;
    const float* safe = reinterpret_cast<const float*>(p.tab);   // 32K floats: what an absent operand reads
    struct Ops {
        float4 a[NV], ab[NV], r[NV], w[NV], b[NV];
        float m;
        uint32_t f;          // the link's scalars, read with its operands
        float eps, scale;
        float *s, *y;
    };
    // every load is unconditional, so those of the links ahead are in flight
    // together while this one reduces
    auto load = [&](int i) __attribute__((always_inline)) {
        Ops o;
        const RowLink& L = p.l[i];
        o.f = L.flags;
        o.eps = L.eps;
        o.scale = L.scale;
        o.s = L.s;
        o.y = L.y;
        arg_now(o.f); arg_now(__builtin_bit_cast(uint32_t, o.eps)); arg_now(__builtin_bit_cast(uint32_t, o.scale));
        arg_now(o.s); arg_now(o.y); arg_now(L.a); arg_now(L.ab); arg_now(L.r); arg_now(L.w); arg_now(L.b); arg_now(L.mask);
        const float* pa = L.a ? L.a + (o.f & kLinkAVec ? 0 : ro) : safe;
        const float* pc = L.ab ? L.ab : safe;
        const float* pr = L.r ? L.r + ro : safe;
        const float* pw = L.w ? L.w : safe;
        const float* pb = L.b ? L.b : safe;
        o.m = *(L.mask ? L.mask + row : safe);
#pragma unroll
        for (int k = 0; k < NV; k++) {
            const int64_t j = (lane + 64 * k) * 4, jc = j < ne0 ? j : 0;
            o.a[k] = *reinterpret_cast<const float4*>(pa + jc);
            o.ab[k] = *reinterpret_cast<const float4*>(pc + jc);
            o.r[k] = *reinterpret_cast<const float4*>(pr + jc);
            o.w[k] = *reinterpret_cast<const float4*>(pw + jc);
            o.b[k] = *reinterpret_cast<const float4*>(pb + jc);
        }
        return o;
    };
    float4 S[NV], Y[NV];   // the last link's sum and result
#pragma unroll
    for (int k = 0; k < NV; k++) S[k] = Y[k] = make_float4(0.f, 0.f, 0.f, 0.f);
    auto step = [&](const Ops o) __attribute__((always_inline)) {
        const uint32_t f = o.f, fa = f >> kLinkA & 3u, fr = f >> kLinkR & 3u;
        float4 v[NV];
#pragma unroll
        for (int k = 0; k < NV; k++) {
            float4 t = o.a[k], q = o.r[k];
            if (fa == kFromSum) t = S[k];
            if (fa == kFromResult) t = Y[k];
            if (fr == kFromSum) q = S[k];
            if (fr == kFromResult) q = Y[k];
            const float4 c = o.ab[k];
            if (f & kLinkBias) t = make_float4(t.x + c.x, t.y + c.y, t.z + c.z, t.w + c.w);
            if (fr != kAbsent) t = make_float4(t.x + q.x, t.y + q.y, t.z + q.z, t.w + q.w);
            const bool in = (lane + 64 * k) * 4 < ne0;
            v[k] = make_float4(in ? t.x : 0.f, in ? t.y : 0.f, in ? t.z : 0.f, in ? t.w : 0.f);
            S[k] = v[k];
        }
        if (o.s) {
#pragma unroll
            for (int k = 0; k < NV; k++) {
                const int64_t j = (lane + 64 * k) * 4;
                if (j < ne0) Stream<float>::store4(reinterpret_cast<char*>(o.s + ro + j), v[k]);
            }
        }
        if (f & kLinkNorm) {
            const float scale = row_scale_w<NV, NORM_LN, WPR>(v, lane, ne0, o.eps, lds);
#pragma unroll
            for (int k = 0; k < NV; k++) {
#pragma unroll
                for (int e = 0; e < 4; e++) set(v[k], e, get(v[k], e) * scale * get(o.w[k], e) + get(o.b[k], e));
            }
            if (f & kLinkMish) apply_act_vec<NV>(CBX_UNARY_MISH, v, p.tab, 0.0f);
        }
        if (f & kLinkMask) {
#pragma unroll
            for (int k = 0; k < NV; k++) v[k] = make_float4(v[k].x * o.m, v[k].y * o.m, v[k].z * o.m, v[k].w * o.m);
        }
        if (f & kLinkScale) {
            const float c = o.scale;
#pragma unroll
            for (int k = 0; k < NV; k++) v[k] = make_float4(v[k].x * c, v[k].y * c, v[k].z * c, v[k].w * c);
        }
#pragma unroll
        for (int k = 0; k < NV; k++) Y[k] = v[k];
        if (o.y) {
#pragma unroll
            for (int k = 0; k < NV; k++) {
                const int64_t j = (lane + 64 * k) * 4;
                if (j < ne0) Stream<float>::store4(reinterpret_cast<char*>(o.y + ro + j), v[k]);
            }
        }
    };
    // the links into the scalar cache, a dozen at a time: met one by one,
    // each would stall its loads on a miss
    static_assert(kChainMax % 12 == 0, "whole dozens");
    for (int i = 0; i < p.n; i += 12) {
        const void* t[24];
#pragma unroll
        for (int q = 0; q < 12; q++) {
            t[2 * q] = p.l[i + q].a;
            t[2 * q + 1] = p.l[i + q].s;
        }
#pragma unroll
        for (int q = 0; q < 24; q++) arg_now(t[q]);
    }
    // three links a turn, each loaded three ahead into registers of its own
    // (the host pads the list to whole turns with links that do nothing)
    Ops o0 = load(0), o1 = load(1), o2 = load(2);
    for (int i = 0; i < p.n; i += 3) {
        const int nx = i + 3 < p.n ? i + 3 : 0;
        step(o0);
        o0 = load(nx);
        step(o1);
        o1 = load(nx + 1);
        step(o2);
        o2 = load(nx + 2);
    }
}

}  // namespace

int launch_elt_group(const EltOp* ops, int n, DeviceState* st, hipStream_t s) {
    for (int i0 = 0; i0 < n; i0 += kEltMax) {
        EltArgs a;
        a.n = std::min(n - i0, kEltMax);
        a.tab = st->gelu_table;
        uint32_t at = 0;
        for (int k = 0; k < a.n; k++) {
            a.op[k] = ops[i0 + k];
            a.first[k] = at;
            at += static_cast<uint32_t>(cdiv(a.op[k].n4, kThreads));
        }
        for (int k = a.n; k < kEltMax; k++) a.first[k] = UINT32_MAX;
        hipLaunchKernelGGL(k_elt_group, dim3(at), dim3(kThreads), 0, s, a);
    }
    return check_launch("elt_group");
}

int launch_row_chain(const RowLink* ls, int n, int64_t ne0, int64_t nr, DeviceState* st, hipStream_t s) {
    static_assert(kChainMax % 3 == 0, "whole turns");
    ChainArgs a;
    a.n = static_cast<int32_t>(cdiv(n, 3) * 3);
    a.ne0 = static_cast<int32_t>(ne0);
    a.tab = st->gelu_table;
    std::copy(ls, ls + n, a.l);
    std::fill(a.l + n, a.l + kChainMax, RowLink{});
    // vectors a lane and waves a row: launch_layer_norm_ext's choice, so each
    // link's reductions add in the same order as its own launch's
    const int nv = ne0 <= 256 ? 1 : ne0 <= 512 ? 2 : 4;
    int wpr = 1;
    while (wpr < 4 && wpr < nv && nr * wpr < int64_t{8} * st->n_cu) wpr *= 2;
    const dim3 grid(static_cast<unsigned>(nr)), block(64 * wpr);
    switch (nv * 8 + wpr) {
        case 1 * 8 + 1: hipLaunchKernelGGL((k_row_chain<1, 1>), grid, block, 0, s, a); break;
        case 2 * 8 + 1: hipLaunchKernelGGL((k_row_chain<2, 1>), grid, block, 0, s, a); break;
        case 2 * 8 + 2: hipLaunchKernelGGL((k_row_chain<1, 2>), grid, block, 0, s, a); break;
        case 4 * 8 + 1: hipLaunchKernelGGL((k_row_chain<4, 1>), grid, block, 0, s, a); break;
        case 4 * 8 + 2: hipLaunchKernelGGL((k_row_chain<2, 2>), grid, block, 0, s, a); break;
        default: hipLaunchKernelGGL((k_row_chain<1, 4>), grid, block, 0, s, a); break;
    }
    return check_launch("row_chain");
}

}  // namespace cbx

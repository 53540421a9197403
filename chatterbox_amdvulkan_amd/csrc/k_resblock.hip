// k_resblock.hip -- one ResBlock layer of the HiFT vocoder,
//   y = res + conv2(snake2(conv1(snake1(x)) + b1)) + b2 [+ the ResBlock sum],
// as one launch (resblock_forward's loop body, hift_vocoder.cpp:119-138), and
// the layers of up to kResMax independent ResBlocks side by side in it.
//
// What bounds the two convs run one by one (k_conv1d.hip): each launch writes
// its f32 output and reads it back, stages and activates a window per output
// tile, and its matrix-core phase waits for the staging and the stores of the
// same launch.  Here a workgroup keeps a tile's intermediate in LDS: it stages
// the activated f16 window of x once, runs conv1 over M frames, activates the
// sums in registers into an f16 window in the same LDS, and runs conv2 on it;
// M - (K2-1)*d2 of the M frames are outputs, the rest is conv2's halo.
//
// Arithmetic class: k_conv1d's.  snake1(x) in f32 rounded to f16 (the im2col
// rounding), f16 products summed in f32 from b1 on, snake2 in f32, rounded to
// f16, f16 products summed in f32 from b2 on, + res [, + sum, * scale].
//
// Operands: the weights are the A operand of v_mfma_f32_32x32x16_f16 (rows =
// output channels) and the window rows the B operand (columns = frames); the
// prepared fragments serve as either, the lane layouts being the same.  A
// lane then holds four consecutive channels of one frame per accumulator
// quad: 8-byte LDS writes of the intermediate and float4 stores of the result
// straight from the accumulators.
//
// Tile: each wave owns MT*32 frames x 32 channels and all of the reduction
// (no partial sums to exchange).  A step (one tap, 16 channels) reads MT KiB
// of LDS and one KiB of weights for MT MFMAs of 32 cycles.  What is left
// besides the matrix cores is the activation (about 22 vector instructions
// an element, twice), the first read of x and the launch itself, so small
// workgroups, several of them on a CU in different phases, beat the larger
// tiles whose steps read less: three layers of 64 x 60001 K 11, 128 x 64
// tiles of 64 x 32 a wave 79.8 us against 86.9 for 256 x 64 tiles of 64 x 64
// a wave; 128 x 20000 K 3, 64 x 128 tiles 53.3 against 67.9 for 128 x 128.
// Against the convs one by one (three layers, us): 64 x 60001 K 3 / 7 / 11
// 54.8 / 66.6 / 76.2 from 72.6 / 87.4 / 101; 128 x 20000 52.8 / 70.3 / 90.3
// from 87.8 / 105 / 126; 256 x 4000 47.8 / 80.5 / 112 from 73.5 / 96.2 / 115.
#include "cbx_device.h"

namespace cbx {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

struct ResArgs {
    int32_t n;
    uint32_t first[kResMax];    // first workgroup of each layer, a multiple of 8
    ResLayer l[kResMax];
};

template <int CH, int MT, int NT, int WM, int WN, int PF>
__global__ __launch_bounds__(64 * WM * WN) __attribute__((amdgpu_waves_per_eu(2))) void k_res_layer(ResArgs a) {
    static_assert(WN * NT * 32 == CH, "a workgroup owns all channels");
    constexpr int NTH = 64 * WM * WN, M = WM * MT * 32, NB = CH / 16, cs = CH + 8;
    static_assert(NB % PF == 0, "ring slots are static");
    extern __shared__ _Float16 lds[];   // window of x (M + (k1-1)*d1 rows of cs halves), then of the intermediate
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave % WN;
    int li = 0;
    if (a.n > 1 && blockIdx.x >= a.first[1]) li = 1;
    if (a.n > 2 && blockIdx.x >= a.first[2]) li = 2;
    const ResLayer p = a.l[li];
    // workgroup L of a layer runs on XCD L % 8 (its first one is a multiple
    // of 8): neighbouring tiles, which share halo rows, on one XCD
    const unsigned L = blockIdx.x - a.first[li], n_wg = static_cast<unsigned>(p.tiles);
    if (L >= n_wg) return;
    const unsigned q8 = n_wg >> 3, r8 = n_wg & 7, xcd = L & 7, j8 = L >> 3;
    const unsigned w = xcd < r8 ? xcd * (q8 + 1) + j8 : r8 * (q8 + 1) + (xcd - r8) * q8 + j8;
    const int pad1 = (p.k1 - 1) * p.d1 / 2, pad2 = (p.k2 - 1) * p.d2 / 2;
    const int mv = M - 2 * pad2;                       // output frames of a tile
    const int t0 = static_cast<int>(w) * mv;
    const int h0 = t0 - pad2;                          // frame of intermediate row 0
    const int base_t = h0 - pad1;                      // frame of window row 0
    const int win = M + 2 * pad1;

    // weights of the first tap (each workgroup starts at its own tap, so the
    // workgroups of an XCD spread their fragment reads over its L2); they
    // arrive while the window is staged
    const int lo = lane * 8;
    const _Float16* wf1 = p.w1 + static_cast<int64_t>(wn * NT) * p.k1 * (NB * 512);
    const _Float16* wf2 = p.w2 + static_cast<int64_t>(wn * NT) * p.k2 * (NB * 512);
    const int ks1 = static_cast<int>(j8 % static_cast<unsigned>(p.k1));
    const int ks2 = static_cast<int>(j8 % static_cast<unsigned>(p.k2));
    half8 ring[PF][NT];
#pragma unroll
    for (int q = 0; q < PF; q++) {
#pragma unroll
        for (int nt = 0; nt < NT; nt++) {
            ring[q][nt] = *reinterpret_cast<const half8*>(wf1 + (static_cast<int64_t>(nt) * p.k1 + ks1) * (NB * 512) +
                                                          q * 512 + lo);
        }
    }

    // the activated window of x as f16
    {
        constexpr int gpr = CH / 4, dr = NTH / gpr, KST = 10;
        const int r0 = tid / gpr, cg = 4 * (tid % gpr);
        const float4 al = *reinterpret_cast<const float4*>(p.al1 + cg);
        const float4 ai = *reinterpret_cast<const float4*>(p.ai1 + cg);
        float mx = 0.0f;
        for (int p0 = 0; p0 * dr < win; p0 += KST) {
            float4 v[KST];
#pragma unroll
            for (int i = 0; i < KST; i++) {
                const int rr = r0 + (p0 + i) * dr, ti = base_t + rr;
                const bool ok = rr < win && ti >= 0 && ti < p.T;
                // rows outside x read row 0 and are zeroed (snake(0) = 0)
                const float4 t = *reinterpret_cast<const float4*>(p.x + static_cast<int64_t>(ok ? ti : 0) * p.x_nb1 +
                                                                  cg * 4);
                v[i] = ok ? t : make_float4(0.f, 0.f, 0.f, 0.f);
            }
#pragma unroll
            for (int i = 0; i < KST; i++) {
                const int rr = r0 + (p0 + i) * dr;
                if (rr < win) {
                    half4 hv;
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        const float xv = get(v[i], q), xa = xv * get(al, q);
                        mx = fmaxf(mx, fabsf(xa));
                        hv[q] = static_cast<_Float16>(xv + sin_sq_small(xa) * get(ai, q));
                    }
                    *reinterpret_cast<half4*>(lds + rr * cs + cg) = hv;
                }
            }
        }
        // rare: this thread's elements with an argument of sin at or past
        // kSinSmall again, with the library sinf
        if (!(mx < kSinSmall)) {
            for (int rr = r0; rr < win; rr += dr) {
                const int ti = base_t + rr;
                if (ti < 0 || ti >= p.T) continue;
                const float* row = reinterpret_cast<const float*>(p.x + static_cast<int64_t>(ti) * p.x_nb1);
                for (int q = 0; q < 4; q++) {
                    lds[rr * cs + cg + q] =
                        static_cast<_Float16>(snake_elem(row[cg + q], p.al1[cg + q], p.ai1[cg + q]));
                }
            }
        }
    }
    __syncthreads();

    floatx16 acc[MT][NT];
    const int lrow = lane & 31, lk = 8 * (lane >> 5);
    int arow[MT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++) arow[mt] = ((wm * MT + mt) * 32 + lrow) * cs + lk;

    // One conv over the window in LDS, its sums starting at the bias: taps from k0 on, cyclically; the
    // weights of step s sit in ring slot s % PF, read PF steps ahead -- past
    // the last tap from wn_ (the next conv's first tap), so no load has a
    // condition; the window rows are read one step ahead.
    const int cbase = wn * NT * 32 + 4 * (lane >> 5);   // accumulator 4g + q of tile nt: channel cbase + 32nt + 8g + q
    auto conv = [&](const _Float16* wf, const float* bias, int k, int d, int k0, const _Float16* wnext, int knext,
                    int k0next) {
#pragma unroll
        for (int nt = 0; nt < NT; nt++) {
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const float4 b4 = *reinterpret_cast<const float4*>(bias + cbase + nt * 32 + 8 * g);
#pragma unroll
                for (int mt = 0; mt < MT; mt++) {
#pragma unroll
                    for (int q = 0; q < 4; q++) acc[mt][nt][4 * g + q] = get(b4, q);
                }
            }
        }
        half8 bv[2][MT];
        int aoff = k0 * d * cs;
#pragma unroll
        for (int mt = 0; mt < MT; mt++) bv[0][mt] = *reinterpret_cast<const half8*>(lds + arow[mt] + aoff);
        int tap = k0;
        const _Float16* wc = wf + static_cast<int64_t>(tap) * (NB * 512);   // this tap's weights, co tile 0
        int64_t cstep = static_cast<int64_t>(k) * (NB * 512);               // to the next co tile
        for (int i = 0; i < k; i++) {
            const int tn = tap + 1 == k ? 0 : tap + 1;
            const bool last = i + 1 == k;
            const int an = last ? aoff : tn * d * cs;      // past the end: unused
            const _Float16* wx = last ? wnext + static_cast<int64_t>(k0next) * (NB * 512)
                                      : wf + static_cast<int64_t>(tn) * (NB * 512);
            const int64_t xstep = last ? static_cast<int64_t>(knext) * (NB * 512) : cstep;
#pragma unroll
            for (int b = 0; b < NB; b++) {
                const int cur = b & 1;
                const int o = b + 1 < NB ? aoff + (b + 1) * 16 : an;
#pragma unroll
                for (int mt = 0; mt < MT; mt++) bv[cur ^ 1][mt] = *reinterpret_cast<const half8*>(lds + arow[mt] + o);
#pragma unroll
                for (int mt = 0; mt < MT; mt++) {
#pragma unroll
                    for (int nt = 0; nt < NT; nt++) {
                        acc[mt][nt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ring[b % PF][nt], bv[cur][mt], acc[mt][nt],
                                                                             0, 0, 0);
                    }
                }
                // the weights of step b + PF
                const _Float16* src = b + PF < NB ? wc + (b + PF) * 512 : wx + (b + PF - NB) * 512;
                const int64_t st = b + PF < NB ? cstep : xstep;
#pragma unroll
                for (int nt = 0; nt < NT; nt++) ring[b % PF][nt] = *reinterpret_cast<const half8*>(src + nt * st + lo);
            }
            tap = tn;
            aoff = an;
            wc = wx;
        }
    };

    conv(wf1, p.b1, p.k1, p.d1, ks1, wf2, p.k2, ks2);
    __syncthreads();   // the window of x has been read

    // snake2 of the sums as f16 intermediate rows, zero outside [0, T)
    // (conv2's padding)
    const bool inner = h0 >= 0 && h0 + M <= p.T;
    float mx = 0.0f;
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const int co = cbase + nt * 32 + 8 * g;
            const float4 al = *reinterpret_cast<const float4*>(p.al2 + co);
            const float4 ai = *reinterpret_cast<const float4*>(p.ai2 + co);
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
                const int row = (wm * MT + mt) * 32 + lrow, t = h0 + row;
                half4 hv;
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const float v = acc[mt][nt][4 * g + q], xa = v * get(al, q);
                    mx = fmaxf(mx, fabsf(xa));
                    hv[q] = static_cast<_Float16>(v + sin_sq_small(xa) * get(ai, q));
                }
                if (!inner && (t < 0 || t >= p.T)) hv = half4{};
                *reinterpret_cast<half4*>(lds + row * cs + co) = hv;
            }
        }
    }
    if (!(mx < kSinSmall)) {
        // rare: the lane's elements one by one with the library sinf; each
        // is picked out of the accumulators by selects (a lane-dynamic
        // register index is not addressable)
        for (int e = 0; e < MT * NT * 16; e++) {
            float v = 0.0f;
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
#pragma unroll
                for (int nt = 0; nt < NT; nt++) {
#pragma unroll
                    for (int r = 0; r < 16; r++) v = e == (mt * NT + nt) * 16 + r ? acc[mt][nt][r] : v;
                }
            }
            const int r = e & 15, nt = (e >> 4) % NT, mt = (e >> 4) / NT;
            const int co = cbase + nt * 32 + 8 * (r >> 2) + (r & 3), row = (wm * MT + mt) * 32 + lrow, t = h0 + row;
            if (t >= 0 && t < p.T) lds[row * cs + co] = static_cast<_Float16>(snake_elem(v, p.al2[co], p.ai2[co]));
        }
    }
    __syncthreads();

    // the residual, read while conv2 runs
    float4 rv[NT][MT][4];
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
            const int t = t0 + (wm * MT + mt) * 32 + lrow;
            const char* rr = p.res + static_cast<int64_t>(t < p.T ? t : p.T - 1) * p.r_nb1 + (cbase + nt * 32) * 4;
#pragma unroll
            for (int g = 0; g < 4; g++) rv[nt][mt][g] = *reinterpret_cast<const float4*>(rr + 32 * g);
        }
    }
    conv(wf2, p.b2, p.k2, p.d2, ks2, wf2, p.k2, ks2);

    // y = res + (sum + b2) [+ the ResBlock sum [* scale]]: the reference's
    // adds in its order; a lane stores four channels of one frame
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
        const int row = (wm * MT + mt) * 32 + lrow, t = t0 + row;
        if (row < mv && t < p.T) {
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    const int co = cbase + nt * 32 + 8 * g;
                    const float4 r = rv[nt][mt][g];
                    const floatx16& c = acc[mt][nt];
                    float4 v = make_float4(r.x + c[4 * g], r.y + c[4 * g + 1], r.z + c[4 * g + 2], r.w + c[4 * g + 3]);
                    if (p.acc) {
                        const float4 s = *reinterpret_cast<const float4*>(p.acc + static_cast<int64_t>(t) * p.a_nb1 +
                                                                          co * 4);
                        v = make_float4(s.x + v.x, s.y + v.y, s.z + v.z, s.w + v.w);
                        if (p.scaled) {
                            v = make_float4(v.x * p.oscale, v.y * p.oscale, v.z * p.oscale, v.w * p.oscale);
                        }
                    }
                    *reinterpret_cast<float4*>(p.y + static_cast<int64_t>(t) * p.y_nb1 + co * 4) = v;
                }
            }
        }
    }
}

}  // namespace

// The variants, one per channel count: M frames a tile, by WM x WN waves of
// MT x 1 MFMA tiles.
template <int CH> struct ResTile;
template <> struct ResTile<64> { static constexpr int MT = 2, WM = 2, WN = 2, PF = 4, M = 128; };
template <> struct ResTile<128> { static constexpr int MT = 2, WM = 1, WN = 4, PF = 8, M = 64; };
template <> struct ResTile<256> { static constexpr int MT = 1, WM = 1, WN = 8, PF = 8, M = 32; };
// 256 channels, when 32-frame tiles are more than 1.5 a CU (the layers of
// three ResBlocks side by side): 64-frame tiles read each weight half as often
struct ResTileWide { static constexpr int MT = 2, WM = 1, WN = 8, PF = 16, M = 64; };

static int64_t res_rows(int ch) {
    return ch == 64 ? ResTile<64>::M : ch == 128 ? ResTile<128>::M : ch == 256 ? ResTile<256>::M : 0;
}

static int64_t res_tiles(const ResLayer& l, int64_t m) {
    const int64_t mv = m - static_cast<int64_t>(l.k2 - 1) * l.d2;
    return mv > 0 ? cdiv(l.T, mv) : 0;
}

static size_t res_lds(const ResLayer& l, int ch, int64_t m) {
    const int64_t rows = m + std::max(static_cast<int64_t>(l.k1 - 1) * l.d1, static_cast<int64_t>(l.k2 - 1) * l.d2);
    return static_cast<size_t>(rows) * static_cast<size_t>(ch + 8) * sizeof(_Float16);
}

// Where one launch beats the two convs one by one: from 1/8 of a tile per CU
// up for short taps, from more for long ones, whose unfused form spreads a
// few frames over more workgroups (three layers, us, fused against not:
// 64 x 12000 K 3 31.6 / 48.0, K 11 45.6 / 52.9, 64 x 6000 K 3 32.9 / 40.6,
// K 11 46.6 / 43.9; 128 x 5000 K 11 58.8 / 72.3, 128 x 2500 K 11 56.0 / 56.2).
// 256 channels read every weight per 32 frames, so K 7 and 11 take more
// tiles to pay (256 x 4000 K 7 80.5 / 96.2, K 11 112 / 115; 256 x 2000 K 3
// 44.8 / 61.5, K 7 78.2 / 76.5, K 11 105 / 92).
bool res_layer_fits(const ResLayer& l, int ch, const DeviceState* st) {
    const int64_t m = res_rows(ch);
    if (m == 0 || res_lds(l, ch, m) > 64 * 1024) return false;
    const int64_t tiles = res_tiles(l, m), k = l.k1 + l.k2, n_cu = st->n_cu;
    // kResMax layers of this many tiles, 512 work-items each: under 2^32 a launch
    if (tiles < 1 || tiles >= (int64_t{1} << 21)) return false;
    if (ch == 256 && k > 6) return k > 14 ? 3 * tiles >= 2 * n_cu : 3 * tiles >= n_cu;
    return (k > 14 ? 3 : 8) * tiles >= n_cu;
}

template <typename R, int CH>
static void res_launch(uint32_t grid, size_t lds, hipStream_t s, const ResArgs& a) {
    static_assert(R::M == R::WM * R::MT * 32, "tile rows");
    hipLaunchKernelGGL((k_res_layer<CH, R::MT, 1, R::WM, R::WN, R::PF>), dim3(grid), dim3(64 * R::WM * R::WN), lds, s, a);
}

int launch_res_layers(const ResLayer* ls, int n, int ch, DeviceState* st, hipStream_t s) {
    ResArgs a;
    a.n = n;
    uint32_t at = 0;
    size_t lds = 0;
    int64_t m = res_rows(ch), tiles = 0;
    for (int i = 0; i < n; i++) tiles += res_tiles(ls[i], m);
    if (ch == 256 && 2 * tiles > int64_t{3} * st->n_cu) {
        bool fits = true;
        for (int i = 0; i < n; i++) fits = fits && res_lds(ls[i], ch, ResTileWide::M) <= 64 * 1024;
        if (fits) m = ResTileWide::M;
    }
    for (int i = 0; i < n; i++) {
        a.l[i] = ls[i];
        a.l[i].tiles = static_cast<int32_t>(res_tiles(ls[i], m));
        a.first[i] = at;
        at += static_cast<uint32_t>(cdiv(a.l[i].tiles, 8) * 8);
        lds = std::max(lds, res_lds(ls[i], ch, m));
    }
    if (ch == 64) res_launch<ResTile<64>, 64>(at, lds, s, a);
    else if (ch == 128) res_launch<ResTile<128>, 128>(at, lds, s, a);
    else if (m == ResTileWide::M) res_launch<ResTileWide, 256>(at, lds, s, a);
    else res_launch<ResTile<256>, 256>(at, lds, s, a);
    return check_launch("res_layers");
}

}  // namespace cbx

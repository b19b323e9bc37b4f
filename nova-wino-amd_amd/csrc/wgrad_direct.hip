// Weight gradient of the 3x3 convolution for float16 output gradients:
//
//   dw[k][c][r][s] = sum over images b and pixels (h, w) of the output
//                    dY[b][k][h][w] * x[b][c][h + r - pad][w + s - pad]
//
// as nine products over the pixels (one per tap), on float16 MFMA with
// float32 accumulation. Both operands are the caller's float16 tensors, so
// every product is exact and only the float32 sums round.
//
// Workgroup: 8 waves, WK x WC x WP of them; the workgroup owns 32*WK output
// channels x 32*WC input channels and one range ("split") of the units; wave
// (wk, wc, wp) holds the nine 32 x 32 taps of its channel pair
// (v_mfma_f32_32x32x16_f16, 144 accumulators) for every WP-th step. A unit is
// R rows of x of G images (G > 1 only for whole images), in a column strip of
// Ws 8-pixel segments, with the R + 2 rows of dY that meet them, in an LDS
// buffer of 16-byte chunks (8 pixels of one channel).
//
// A step multiplies two segments (16 pixels: lanes 0-31 hold one, lanes 32-63
// the next; each lane 8 consecutive pixels of its channel). x is owned by
// row, and the three taps r pair one x row with three dY rows, so a step
// reads one x segment with the halves left and right of it, shifts it by one
// pixel either way in registers (v_alignbyte), and reads three dY segments:
// 4 16-byte LDS reads for 9 MFMAs. Rows of x outside the image are no work;
// other pixels outside it are zeros in LDS, so a lane never multiplies a
// neighbouring row's or channel's value, and an infinity stays in its own
// channel's taps.
//
// Staging: where every row starts on a dword (even widths) the chunks go from
// memory to LDS directly (buffer_load ... lds, no registers), three buffers,
// two units ahead; a last chunk that reaches into the next row is masked when
// it is read. Odd widths go through registers, shifted and masked there, two
// buffers, one unit ahead.
// What bounds it: a unit's fixed costs, not the matrix cores or memory. At
// 64@56^2 batch 32 a turn of the loop takes 3 500 cycles for 1 150 cycles of
// MFMA: issuing a wave's 7 direct loads takes 700, the first fragment reads
// after the barrier about 500, and the two waves of a SIMD overlap the rest.
// Without the loads the launch is 5 % faster, without the products 25 %.
//
// Measured on MI355X (whole nova_weight_grad, us, the float32 Winograd-domain
// form of wgrad.hip -> this one): ResNet-50 batch 32 64@56^2 91.7 -> 27.5,
// 128@28^2 65.1 -> 30.4, 256@14^2 71.7 -> 29.4, 512@7^2 94.5 -> 29.7;
// 320@64^2 batch 8 361 -> 84.8 (712 TFLOP/s). Relative error against float64
// 1.2e-5 - 1.6e-5 -> 1e-7 - 3e-7 (no transform, exact products).
#include <algorithm>

#include "nova_internal.h"
#include "nova_tile_math.h"

namespace nova {

namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f16v __attribute__((ext_vector_type(16)));
typedef unsigned u4 __attribute__((ext_vector_type(4)));

constexpr int kThreads = 512;
constexpr int kBufBytes = 52 * 1024;      // one of three LDS buffers
constexpr int kSlots = 7;                 // 16-byte chunks staged per thread and unit
constexpr int kOob = (int)0x80000000;     // out-of-range byte offset: loads 0, stores dropped

// How rows reach LDS: through registers (odd widths), directly, directly with
// masks on a row's last chunk.
enum Stage { kRegs, kDirect, kDirectTail };

struct WdArgs {
    const char* x;
    const char* dy;
    float* out;             // dw, or the splits' partial filters
    float* bias;            // sums of dY: db, or the splits' partial sums; null: none
    int64_t x_bytes, dy_bytes;
    int B, C, K, H, W, Ho, Wo;
    int G, R, nrb;          // images and x rows per unit, row blocks per image
    int Ws, nstrip;         // segments per strip, strips per row
    int lo, XS, XP;         // x row in LDS: left halo chunks, staged chunks, pitch (chunks)
    int xpitch, dpitch;     // chunks per channel in LDS (odd)
    int dstart, zero, nblk; // first dY chunk, first zero chunk, 64-chunk blocks of a unit
    int nwx;                // waves that stage x (the others stage dY)
    unsigned mxp, mdp, mXP, mWs, mR, mR2;  // 2^20 / d + 1 (mxp, mdp), 65536 / d + 1
    int ntk, nt;            // 32*WK-row tiles of K, tiles in all
    int nunits, nsplit;
    int nwg;
};

// t / d for t < 256 and d <= 256 (m = 65536 / d + 1).
__device__ __forceinline__ int fdiv(int t, unsigned m) { return (int)(((unsigned)t * m) >> 16); }

// A buffer resource from p (a multiple of 4) over n bytes, rounded up to the
// dword that holds the last one.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc_of(const char* p, int64_t n) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(p), (short)0,
                                             (int)((n + 3) & ~(int64_t)3), 0x00020000);
}

// t / d for t < 4096 and d <= 256 (m = 2^20 / d + 1).
__device__ __forceinline__ int fdiv20(int t, unsigned m) { return (int)(((unsigned)t * m) >> 20); }

template <int PAD, int WK, int WC, int kStage>
__global__ __launch_bounds__(kThreads) void wgrad_direct_kernel(WdArgs a) {
    constexpr int WP = 8 / (WK * WC);
    // three arrays and not one, each named by its own code: the compiler
    // tells them apart and does not wait for a direct load into one before a
    // read of another
    __shared__ __align__(1024) char buf0[kBufBytes];
    __shared__ __align__(1024) char buf1[kBufBytes];
    __shared__ __align__(1024) char buf2[kBufBytes];
    __shared__ __align__(1024) char spare[1024];  // slots without a block load zeros here
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wk = wave % WK, wc = (wave / WK) % WC, wp = wave / (WK * WC);
    const int L = xcd_remap((int)blockIdx.x, a.nwg);
    const int tile = L % a.nt, sp = L / a.nt;
    const int k0 = (tile % a.ntk) * (32 * WK), c0 = (tile / a.ntk) * (32 * WC);
    const int u_lo = (int)((int64_t)sp * a.nunits / a.nsplit);
    const int nu = (int)((int64_t)(sp + 1) * a.nunits / a.nsplit) - u_lo;
    const int HW = a.H * a.W, HoWo = a.Ho * a.Wo;

    // A unit's row block, column strip and image group (advanced without
    // divisions).
    struct Unit {
        int rb, strip, g;
    };
    auto advance = [&](Unit& n) {
        if (++n.rb < a.nrb) return;
        n.rb = 0;
        if (++n.strip == a.nstrip) {
            n.strip = 0;
            n.g++;
        }
    };
    Unit ul, up;  // next unit to load, next to multiply
    {
        const int t = u_lo / a.nrb;
        ul.rb = u_lo - t * a.nrb;
        ul.g = t / a.nstrip;
        ul.strip = t - ul.g * a.nstrip;
        up = ul;
    }

    // Staging: the unit's LDS image is x chunks (channel-major), dY chunks
    // from dstart on and zeros from `zero` on, in 64-chunk blocks, one block a
    // wave and slot; nwx waves take the x blocks, the others the dY blocks, so
    // a wave has one resource, one row length and one set of bounds. A chunk's
    // byte offset from its unit's first row (off, kOob where it is always
    // zeros) and its dY row and its segment (pos: bits 0-7 and 8-15) do not
    // change between units. The resource starts above the first row that a
    // unit may name (dY's halo rows, x's left halo chunk), which is never
    // loaded.
    const bool is_x = wave < a.nwx;
    const int nwav = is_x ? a.nwx : 8 - a.nwx, wav = is_x ? wave : wave - a.nwx;
    const int blk0 = (is_x ? 0 : a.dstart >> 6) + wav;
    const int nslot = ((is_x ? a.dstart >> 6 : a.nblk) - blk0 + nwav - 1) / nwav;
    const int row_len = is_x ? a.W : a.Wo;
    const int lead = 2 * (is_x ? 8 * a.lo : (2 - PAD) * a.Wo);
    const int chan0 = is_x ? c0 * HW : k0 * HoWo;
    const char* const src = (is_x ? a.x : a.dy) + 2 * (int64_t)chan0 - lead;
    const int odd = (int)(reinterpret_cast<uint64_t>(src) & 2);
    const __amdgpu_buffer_rsrc_t rs =
        rsrc_of(src - odd, (is_x ? a.x_bytes : a.dy_bytes) - 2 * (int64_t)chan0 + lead + odd);
    const int img_bytes = 2 * a.G * (is_x ? a.C * HW : a.K * HoWo);
    // byte offset of a unit's first row (and left halo chunk)
    auto unit_off = [&](const Unit& n) {
        return n.g * img_bytes + 2 * (n.rb * a.R * row_len + 8 * n.strip * a.Ws) + odd;
    };
    int off[kSlots], pos[kSlots];
#pragma unroll
    for (int s = 0; s < kSlots; s++) {
        off[s] = kOob;
        pos[s] = 0;
        if (s >= nslot) continue;
        const int n = (blk0 + s * nwav) * 64 + lane;
        if (is_x) {
            const int cl = fdiv20(n, a.mxp), t = n - cl * a.xpitch - 1;
            const int rr = t < 0 ? 0 : fdiv(t, a.mXP), i = t - rr * a.XP;
            const int img = fdiv(rr, a.mR), row = rr - img * a.R;
            pos[s] = i << 8;
            if (cl < 32 * WC && c0 + cl < a.C && t >= 0 && i < a.XS && img < a.G)
                off[s] = 2 * (img * a.C * HW + cl * HW + row * a.W + 8 * i);
        } else {
            const int m = n - a.dstart;
            const int cl = fdiv20(m, a.mdp), t = m - cl * a.dpitch;
            const int dr = fdiv(t, a.mWs), i = t - dr * a.Ws;
            const int img = fdiv(dr, a.mR2), row = dr - img * (a.R + 2);
            // one row block: every unit has the same rows outside the image
            const int ho = row + PAD - 2;
            const bool in = a.nrb > 1 || (ho >= 0 && ho < a.Ho);
            pos[s] = row | i << 8;
            if (n < a.zero && cl < 32 * WK && k0 + cl < a.K && img < a.G && in)
                off[s] = 2 * (img * a.K * HoWo + cl * HoWo + row * a.Wo + 8 * i);
        }
    }
    const bool check = a.nrb > 1 || a.nstrip > 1;

    u4 sv[kSlots];
    unsigned se[kSlots];
    // Requests the next unit's chunks, always kSlots loads: straight into buf,
    // or into registers.
    auto load_unit = [&](char* buf) {
        const int so = unit_off(ul);
        auto get = [&](int s, int o) {
            if constexpr (kStage == kRegs) {
                o = (o + (so & 2)) & ~3;
                sv[s] = __builtin_amdgcn_raw_buffer_load_b128(rs, o, so & ~3, 0);
                se[s] = __builtin_amdgcn_raw_buffer_load_b32(rs, o + 16, so & ~3, 0);
            } else {
                char* dst = s < nslot ? buf + (blk0 + s * nwav) * 1024 : spare;
                load_lds16(rs, dst, o, so);
            }
        };
        if (check) {
            // rows of dY and segments that lie in the image
            const int q0 = ul.strip * a.Ws - (is_x ? a.lo : 0), ho0 = ul.rb * a.R + PAD - 2;
            const int i_lo = max(0, -q0), i_n = ((row_len + 7) >> 3) - q0 - i_lo;
            const int r_lo = is_x ? 0 : max(0, -ho0);
            const int r_n = is_x ? 1 : min(a.R + 2, a.Ho - ho0) - r_lo;
#pragma unroll
            for (int s = 0; s < kSlots; s++)
                get(s, (unsigned)((pos[s] & 255) - r_lo) < (unsigned)r_n &&
                               (unsigned)((pos[s] >> 8) - i_lo) < (unsigned)i_n
                           ? off[s]
                           : kOob);
        } else {
#pragma unroll
            for (int s = 0; s < kSlots; s++) get(s, off[s]);
        }
        advance(ul);
    };
    // Registers to LDS, shifted to the row's start and cleared past its end.
    auto store_unit = [&](const Unit& n, char* buf) {
        const int so = unit_off(n);
        const int len = row_len + (is_x ? 8 * a.lo : 0) - 8 * n.strip * a.Ws;
        // through an empty asm: as loop invariants the slots' branch
        // conditions would each stay in a pair of scalar registers, and spill
        int ns = nslot;
        asm volatile("" : "+s"(ns));
#pragma unroll
        for (int s = 0; s < kSlots; s++) {
            if (s >= ns) break;
            const unsigned w[5] = {sv[s][0], sv[s][1], sv[s][2], sv[s][3], se[s]};
            const int sh = (off[s] + so) & 2, nv = len - 8 * (pos[s] >> 8);
            u4 v;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                v[i] = __builtin_amdgcn_alignbyte(w[i + 1], w[i], sh);
                v[i] = nv >= 2 * i + 2 ? v[i] : nv == 2 * i + 1 ? v[i] & 0xffffu : 0u;
            }
            *reinterpret_cast<u4*>(buf + ((blk0 + s * nwav) * 64 + lane) * 16) = v;
        }
    };

    f16v acc[9];
#pragma unroll
    for (int t = 0; t < 9; t++)
#pragma unroll
        for (int e = 0; e < 16; e++) acc[t][e] = 0.0f;

    // sums of dY: waves of the first input-channel tile, each lane its row's
    // pixels of the steps it multiplies (tap r = 1 meets every dY row once)
    const bool sums = PAD < 2 && a.bias != nullptr && c0 == 0 && wc == 0;
    float bsum[2] = {0.0f, 0.0f}, bunit = 0.0f;  // a unit's, all units'

    const int l32 = lane & 31, g = lane >> 5;
    const int xrow = (wc * 32 + l32) * a.xpitch + 1 + a.lo;
    const int drow = a.dstart + (wk * 32 + l32) * a.dpitch;
    // Multiplies unit up. x rows past the image and images past the batch are
    // staged but never multiplied.
    auto products = [&](const char* buf) {
        const int rows = a.G > 1 ? min(a.G, a.B - up.g * a.G) * a.R : min(a.R, a.H - up.rb * a.R);
        const int items = rows * a.Ws;
        const int col0 = 8 * up.strip * a.Ws;
        struct Frag {
            unsigned w[6];  // halves -2 .. 9 around the x segment
            u4 d[3];        // dY segments of taps r
        };
        auto read = [&](Frag& f, int st) {
            const int it = 2 * st + g;
            const int rr = fdiv(it, a.mWs), seg = it - rr * a.Ws;
            const int img = fdiv(rr, a.mR);
            const bool ok = it < items;
            const int xo = 16 * (ok ? xrow + rr * a.XP + seg : a.zero + 1);
            const int eo = 16 * (ok ? drow + (rr + 2 * img) * a.Ws + seg : a.zero);
            if (PAD > 0) f.w[0] = *reinterpret_cast<const unsigned*>(buf + xo - 4);
            const u4 m = *reinterpret_cast<const u4*>(buf + xo);
#pragma unroll
            for (int i = 0; i < 4; i++) f.w[i + 1] = m[i];
            if (PAD < 2) f.w[5] = *reinterpret_cast<const unsigned*>(buf + xo + 16);
#pragma unroll
            for (int r = 0; r < 3; r++)
                f.d[r] = *reinterpret_cast<const u4*>(buf + eo + 16 * (2 - r) * a.Ws);
            if constexpr (kStage == kDirectTail) {
                const int col = col0 + 8 * seg;
                // the halves left of the first empty segment of a last strip
                // are the tail of the row's last chunk
                if (PAD > 0) f.w[0] = col - 2 < a.W ? f.w[0] : 0u;
#pragma unroll
                for (int i = 1; i < 6; i++) f.w[i] = col + 2 * (i - 1) < a.W ? f.w[i] : 0u;
#pragma unroll
                for (int i = 0; i < 4; i++)
#pragma unroll
                    for (int r = 0; r < 3; r++) f.d[r][i] = col + 2 * i < a.Wo ? f.d[r][i] : 0u;
            }
        };
        auto multiply = [&](const Frag& f) {
            if (sums) {
#pragma unroll
                for (int i = 0; i < 8; i++) bsum[i & 1] += (float)__builtin_bit_cast(h8, f.d[1])[i];
            }
#pragma unroll
            for (int s = 0; s < 3; s++) {
                // halves s - PAD .. s - PAD + 7 around the segment
                const int first = 2 + s - PAD;
                u4 v;
#pragma unroll
                for (int i = 0; i < 4; i++)
                    v[i] = (first & 1) ? __builtin_amdgcn_alignbyte(f.w[(first >> 1) + i + 1],
                                                                    f.w[(first >> 1) + i], 2)
                                       : f.w[(first >> 1) + i];
                const h8 xv = __builtin_bit_cast(h8, v);
#pragma unroll
                for (int r = 0; r < 3; r++)
                    acc[3 * r + s] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                        __builtin_bit_cast(h8, f.d[r]), xv, acc[3 * r + s], 0, 0, 0);
            }
        };
        if constexpr (kStage == kRegs) {  // no registers to read ahead
            for (int st = wp; 2 * st < items; st += WP) {
                Frag f;
                read(f, st);
                multiply(f);
            }
        } else {
            // the next step's reads in flight during a step's products
            Frag f0, f1;
            int st = wp;
            if (2 * st < items) read(f0, st);
            while (2 * st < items) {
                st += WP;
                if (2 * st < items) read(f1, st);
                __builtin_amdgcn_sched_barrier(0);
                multiply(f0);
                if (2 * st >= items) break;
                st += WP;
                if (2 * st < items) read(f0, st);
                __builtin_amdgcn_sched_barrier(0);
                multiply(f1);
            }
        }
        if (sums) {
            bunit += bsum[0] + bsum[1];
            bsum[0] = bsum[1] = 0.0f;
        }
        advance(up);
    };
    if constexpr (kStage == kRegs) {
        Unit us = ul;
        auto turn = [&](int i, char* cur, char* nxt) {
            if (i + 1 < nu) load_unit(nxt);
            __builtin_amdgcn_sched_barrier(0);
            products(cur);
            __builtin_amdgcn_sched_barrier(0);
            if (i + 1 < nu) {
                store_unit(us, nxt);
                advance(us);
            }
            lds_barrier();
        };
        if (nu > 0) {
            load_unit(buf0);
            store_unit(us, buf0);
            advance(us);
        }
        lds_barrier();
        for (int i = 0; i < nu; i += 2) {
            turn(i, buf0, buf1);
            if (i + 1 < nu) turn(i + 1, buf1, buf0);
        }
    } else {
        // unit i: its loads are over (those of unit i + 1 may be in flight);
        // the barrier also ends unit i - 1's products, whose buffer unit
        // i + 2 is then loaded into. The second wave of each SIMD requests
        // its loads after its products and not before them, so that one wave
        // multiplies while the other issues.
        const bool late = wave >= 4;
        auto turn = [&](int i, char* cur, char* nxt2) {
            if (i + 1 < nu)
                wait_vmcnt<kSlots>();
            else
                wait_vmcnt<0>();
            lds_barrier();
            if (!late && i + 2 < nu) load_unit(nxt2);
            __builtin_amdgcn_sched_barrier(0);
            products(cur);
            __builtin_amdgcn_sched_barrier(0);
            if (late && i + 2 < nu) load_unit(nxt2);
        };
        if (nu > 0) load_unit(buf0);
        if (nu > 1) load_unit(buf1);
        for (int i = 0; i < nu; i += 3) {
            turn(i, buf0, buf2);
            if (i + 1 < nu) turn(i + 1, buf1, buf0);
            if (i + 2 < nu) turn(i + 2, buf2, buf1);
        }
        lds_barrier();
    }

    // The WP waves' sums, a quarter of every tile at a time (8 output
    // channels x 32 input channels x 9 taps), three taps in each buffer:
    // [tap][wave][e][lane], the taps 8 dwords apart in the banks.
    // Accumulator 4*q + e of a lane: output channel 8*q + 4*(lane / 32) + e,
    // input channel lane % 32. Threads then walk dw's own order.
    constexpr int kTapPitch = 8 * 256 + 8;  // dwords
    float* const red[3] = {reinterpret_cast<float*>(buf0), reinterpret_cast<float*>(buf1),
                           reinterpret_cast<float*>(buf2)};
    float* const out = a.out + (int64_t)sp * a.K * a.C * 9;
    if (PAD < 2 && a.bias != nullptr && c0 == 0) {
        if (wc == 0) red[0][wave * 64 + lane] = bunit;
        lds_barrier();
        if (tid < 32 * WK && k0 + tid < a.K) {
            const int w0 = tid >> 5;  // the wave with this row, wc = 0 and wp = 0
            float v = 0.0f;
            for (int p = 0; p < WP; p++) {
                const float* r = red[0] + (w0 + p * WK * WC) * 64 + (tid & 31);
                v += r[0];
                v += r[32];
            }
            a.bias[(int64_t)sp * a.K + k0 + tid] = v;
        }
        lds_barrier();
    }
#pragma unroll
    for (int q = 0; q < 4; q++) {
#pragma unroll
        for (int t = 0; t < 9; t++)
#pragma unroll
            for (int e = 0; e < 4; e++)
                red[t / 3][(t % 3) * kTapPitch + (wave * 4 + e) * 64 + lane] = acc[t][4 * q + e];
        lds_barrier();
        for (int i = tid; i < WK * WC * 8 * 288; i += kThreads) {
            // dw row of pair `pair`: 32 input channels x 9 taps
            const int rowi = i / 288, j = i - rowi * 288;
            const int c = j / 9, tap = j - c * 9;
            const int pair = rowi >> 3, k = rowi & 7;
            const int cc = c0 + 32 * (pair / WK) + c, kk = k0 + 32 * (pair % WK) + 8 * q + k;
            const int o = (tap % 3) * kTapPitch + (pair * 4 + (k & 3)) * 64 + 32 * (k >> 2) + c;
            const float* r = tap < 3 ? red[0] : tap < 6 ? red[1] : red[2];
            float v = r[o];
#pragma unroll
            for (int p = 1; p < WP; p++) v += r[o + p * WK * WC * 256];
            if (cc < a.C && kk < a.K) out[((int64_t)kk * a.C + cc) * 9 + tap] = v;
        }
        lds_barrier();
    }
}

// dw[i] = sum over splits of part[s][i], in split order, for n filter entries
// and then nb bias entries (bpart[s][i] into db).
constexpr int kRedThreads = 256;
__global__ __launch_bounds__(kRedThreads) void wgrad_direct_reduce_kernel(
    const float* __restrict__ part, float* __restrict__ dw, const float* __restrict__ bpart,
    float* __restrict__ db, int64_t n, int nb, int nsplit) {
    const int64_t i = (int64_t)blockIdx.x * kRedThreads + threadIdx.x;
    if (i >= n + nb) return;
    const bool filter = i < n;
    const float* p = filter ? part + i : bpart + (i - n);
    const int64_t ld = filter ? n : nb;
    float v = 0.0f;
    int s = 0;
    for (; s + 16 <= nsplit; s += 16) {
        float r[16];
#pragma unroll
        for (int u = 0; u < 16; u++) r[u] = p[(s + u) * ld];
#pragma unroll
        for (int u = 0; u < 16; u++) v += r[u];
    }
    for (; s + 4 <= nsplit; s += 4) {
        float r[4];
#pragma unroll
        for (int u = 0; u < 4; u++) r[u] = p[(s + u) * ld];
#pragma unroll
        for (int u = 0; u < 4; u++) v += r[u];
    }
    for (; s < nsplit; s++) v += p[s * ld];
    (filter ? dw[i] : db[i - n]) = v;
}

// db[k] = sum of dY[b][k][:] over images and pixels, in fp64, rounded once.
// A channel's pixels are `items` runs of at most kBiasRun of one image, each
// summed by one wave: single elements up to the first 16-byte boundary and
// behind the last, 16-byte loads between, four in flight. nsplit workgroups
// share a channel, each a contiguous range of its runs; their partial sums
// are added by bias_join_kernel (part null: one workgroup, into db).
// Bound by reading dY once. Measured on MI355X beside nova_weight_grad (us, one
// workgroup per channel with 2-byte loads -> this, torch's conversion and sum):
// fp16 32 channels of 64 x 114^2 855 -> 13, 251; 3 of 16 x 514^2 6050 -> 27, 38;
// 320 of 8 x 66^2 42 -> 5, 28; 512 of 32 x 9^2 7 -> 8, 14; fp32 32 of 64 x 112^2
// 1270 -> 25, 219.
constexpr int kBiasThreads = 512, kBiasRun = 8192;
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) v += __shfl_down(v, d, 64);
    return v;
}
template <typename T>
__global__ __launch_bounds__(kBiasThreads) void bias_grad_kernel(
    const T* __restrict__ dy, float* __restrict__ db, double* __restrict__ part, int K,
    int64_t HoWo, int runs, int64_t items, int nsplit) {
    constexpr int kE = 16 / sizeof(T), kWaves = kBiasThreads / 64;
    typedef T vec __attribute__((ext_vector_type(kE)));
    __shared__ double s[kWaves];
    const int k = (int)blockIdx.x / nsplit, sp = (int)blockIdx.x - k * nsplit;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t j = (int64_t)sp * kWaves + wave, nj = (int64_t)nsplit * kWaves;
    double v = 0.0;
    for (int64_t it = j * items / nj; it < (j + 1) * items / nj; it++) {
        const int64_t b = it / runs, at = (it - b * runs) * kBiasRun;
        const int n = (int)min((int64_t)kBiasRun, HoWo - at);
        const T* const p = dy + (b * K + k) * HoWo + at;
        const int to16 = (int)((0 - reinterpret_cast<uintptr_t>(p)) & 15) / (int)sizeof(T);
        const int head = min(to16, n), nv = (n - head) / kE, tail = n - head - nv * kE;
        const vec* const q = reinterpret_cast<const vec*>(p + head);
        if (lane < head) v += (double)p[lane];
        if (lane < tail) v += (double)p[n - tail + lane];
        for (int i = lane; i < nv; i += 256) {
            vec r[4];
#pragma unroll
            for (int u = 0; u < 4; u++) r[u] = q[min(i + 64 * u, nv - 1)];
#pragma unroll
            for (int u = 0; u < 4; u++)
                if (i + 64 * u < nv)
#pragma unroll
                    for (int e = 0; e < kE; e++) v += (double)r[u][e];
        }
    }
    v = wave_sum(v);
    if (lane == 0) s[wave] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        v = s[0];
        for (int w = 1; w < kWaves; w++) v += s[w];
        if (part != nullptr)
            part[blockIdx.x] = v;
        else
            db[k] = (float)v;
    }
}

// db[k] = sum of a channel's nsplit partial sums; one wave per channel.
__global__ __launch_bounds__(256) void bias_join_kernel(const double* __restrict__ part,
                                                        float* __restrict__ db, int K,
                                                        int nsplit) {
    const int k = (int)blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (k >= K) return;
    double v = 0.0;
    for (int i = lane; i < nsplit; i += 64) v += part[(int64_t)k * nsplit + i];
    v = wave_sum(v);
    if (lane == 0) db[k] = (float)v;
}

inline int ceil_div(int a, int b) { return (a + b - 1) / b; }
inline unsigned magic(int d) { return 65536u / (unsigned)d + 1u; }

}  // namespace

// Fills the geometry of one wave arrangement; false where it does not fit.
static bool fill_plan(WgradDirectPlan* p, int B, int C, int K, int H, int W, int pad, int wk,
                      int wc, int G, int R, int Ws) {
    const int Wo = W + 2 * pad - 2;
    const int wseg = ceil_div(Wo, 8), xseg = ceil_div(W, 8);
    p->wk = wk;
    p->wc = wc;
    p->G = G;
    p->R = R;
    p->Ws = Ws;
    p->nrb = ceil_div(H, R);
    if (G > 1 && (R != H || Ws < wseg)) return false;
    p->nstrip = ceil_div(wseg, Ws);
    if (p->nstrip == 1) {
        // one zero chunk between rows is the right pad of one and the left
        // pad of the next
        p->lo = 0;
        p->XS = xseg;
        p->XP = std::max(xseg, Ws) + 1;
    } else {
        p->lo = 1;
        p->XS = Ws + 2;
        p->XP = Ws + 2;
    }
    p->xpitch = (1 + G * R * p->XP) | 1;
    p->dpitch = (G * (R + 2) * Ws) | 1;
    if (p->xpitch > 255 || p->dpitch > 255) return false;
    p->dstart = (32 * wc * p->xpitch + 63) & ~63;
    p->zero = p->dstart + 32 * wk * p->dpitch;
    p->nblk = (p->zero + 2 * Ws + 3 + 63) / 64;
    if (1024 * p->nblk > kBufBytes) return false;
    // waves that stage x: the fewest slots per wave
    int best = kSlots + 1;
    for (int nwx = 1; nwx < 8; nwx++) {
        const int ns = std::max(ceil_div(p->dstart / 64, nwx),
                                ceil_div(p->nblk - p->dstart / 64, 8 - nwx));
        if (ns < best) {
            best = ns;
            p->nwx = nwx;
        }
    }
    if (best > kSlots) return false;
    p->ntk = ceil_div(K, 32 * wk);
    p->nt = p->ntk * ceil_div(C, 32 * wc);
    p->nunits = ceil_div(B, G) * p->nstrip * p->nrb;
    return true;
}

// The arrangement (waves, unit, splits) with the least estimated time, in us:
// rounds of workgroups over the CUs (one each: LDS), each its units and 3 us
// of sums; a unit's two waves per SIMD at 330 cycles a step, or its staging
// (18 cycles per 1 KB block), and 500 cycles for its barrier and first reads;
// splits cost the reduction launch and their partial filters' bytes. One
// round of splits: twice as many workgroups lost everywhere (64@56^2 batch 32
// 28.0 -> 38.5 us, 256@14^2 27.9 -> 39.2). 32 x 32 channels per workgroup up
// to 512 channels at the ResNet-50 shapes (64 x 64 there: 41.5, 41.9, 44.5
// us), larger tiles from 320@64^2 batch 8 on (32 x 32 98.0, 32 x 64 87.8) and
// 64 x 64 where 32 x 64 fills more than one round (1280 -> 640@32^2 batch 2
// 83.3, 66.7 and 57.1; 1280@16^2 82.3, 74.0 and 59.1).
WgradDirectPlan wgrad_direct_plan(int B, int C, int K, int H, int W, int pad, int cus) {
    WgradDirectPlan best{};
    best.ok = false;
    const int Ho = H + 2 * pad - 2, Wo = W + 2 * pad - 2;
    // pads of 3 and more have taps that reach past the halo
    if (pad > 2 || B < 1) return best;
    // 32-bit byte offsets into x and dY, and both resources, each with the
    // rows or the chunk it starts above its tensor, end below kOob (64 bytes
    // for the start's offset, the last dword and a register load's reach)
    const int64_t img = 2 * std::max((int64_t)C * H * W, (int64_t)K * Ho * Wo);
    const int64_t lead = std::max<int64_t>(16, 2 * (2 - pad) * (int64_t)Wo);
    if (B * img + lead > ((int64_t)1 << 31) - 64) return best;
    const int wseg = ceil_div(Wo, 8);
    double best_t = 0.0;
    for (int v = 0; v < 3; v++) {
        const int wk = v == 2 ? 2 : 1, wc = v >= 1 ? 2 : 1, wp = 8 / (wk * wc);
        for (int Ws = std::min(wseg, 16);; Ws = wseg) {
            for (int R = std::min(H, 254 / (Ws + 1)); R >= 1; R--) {
                const int nrb = ceil_div(H, R);
                if (ceil_div(H, nrb) != R) continue;  // even row blocks only
                for (int G = 1; G <= (nrb == 1 ? std::min(B, 16) : 1); G++) {
                    WgradDirectPlan p{};
                    if (!fill_plan(&p, B, C, K, H, W, pad, wk, wc, G, R, Ws)) continue;
                    // splits: one round of workgroups over the CUs
                    int64_t ns = std::max<int64_t>(1, cus / p.nt);
                    ns = std::min<int64_t>(ns, p.nunits);
                    while (ns > 1 && 4 * ns * K * (9 * (int64_t)C + 1) >= ((int64_t)1 << 31)) ns--;
                    p.nsplit = (int)ns;
                    const double rounds =
                        ceil_div((int)std::min<int64_t>(p.nt * ns, 1 << 30), cus);
                    const double units = ceil_div(p.nunits, (int)ns);
                    const double steps = ceil_div(ceil_div(G * R * Ws, 2), wp);
                    const double unit =
                        std::max(2 * steps * 330.0, 18.0 * p.nblk + 400.0) + 500.0;
                    const double part = ns > 1 ? 4.0 + 18e-6 * ns * K * C : 0.0;
                    const double t = rounds * (units * unit / 2.4e3 + 3.0) + part;
                    if (!best.ok || t < best_t) {
                        best = p;
                        best.ok = true;
                        best_t = t;
                    }
                }
            }
            if (Ws == wseg) break;
        }
    }
    // pad 2: no tap meets every dY row
    best.bias = best.ok && pad < 2;
    if (best.ok)
        best.ws_bytes = best.nsplit > 1 ? 4 * (int64_t)best.nsplit * K * (9 * (int64_t)C + 1) : 0;
    return best;
}

template <int PAD, int WK, int WC>
static hipError_t launch_direct(const WdArgs& a, int stage, hipStream_t s) {
    const dim3 grid((unsigned)a.nwg), block(kThreads);
    if (stage == kRegs)
        launch(wgrad_direct_kernel<PAD, WK, WC, kRegs>, grid, block, s, a);
    else if (stage == kDirect)
        launch(wgrad_direct_kernel<PAD, WK, WC, kDirect>, grid, block, s, a);
    else
        launch(wgrad_direct_kernel<PAD, WK, WC, kDirectTail>, grid, block, s, a);
    return hipGetLastError();
}

template <int PAD>
static hipError_t launch_pad(const WdArgs& a, const WgradDirectPlan& p, int stage,
                             hipStream_t s) {
    if (p.wc == 1) return launch_direct<PAD, 1, 1>(a, stage, s);
    if (p.wk == 1) return launch_direct<PAD, 1, 2>(a, stage, s);
    return launch_direct<PAD, 2, 2>(a, stage, s);
}

template <typename T>
static hipError_t launch_bias(const void* dy, float* db, int B, int C, int K, int64_t HoWo,
                              float* dw, int cus, hipStream_t s) {
    // Splits: four workgroups per CU in all, at least one run per wave, and as
    // many fp64 partial sums as dw holds; channels of up to 16384 values are
    // one workgroup's, without the second launch.
    const int64_t runs = (HoWo + kBiasRun - 1) / kBiasRun, items = B * runs;
    int64_t ns = 1;
    if (B * HoWo > 2 * kBiasRun) {
        constexpr int kWaves = kBiasThreads / 64;
        ns = std::min<int64_t>((4 * (int64_t)cus + K - 1) / K, (items + kWaves - 1) / kWaves);
        ns = std::max<int64_t>(1, std::min<int64_t>(ns, (9 * (int64_t)C - 1) / 2));
    }
    double* const part =
        ns > 1 ? reinterpret_cast<double*>((reinterpret_cast<uintptr_t>(dw) + 7) & ~(uintptr_t)7)
               : nullptr;
    launch(bias_grad_kernel<T>, dim3((unsigned)(K * ns)), dim3(kBiasThreads), s,
           static_cast<const T*>(dy), db, part, K, HoWo, (int)runs, items, (int)ns);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || ns == 1) return e;
    launch(bias_join_kernel, dim3((unsigned)((K + 3) / 4)), dim3(256), s,
           static_cast<const double*>(part), db, K, (int)ns);
    return hipGetLastError();
}

hipError_t launch_bias_grad(const void* dy, bool dy_f32, float* db, int B, int C, int K,
                            int64_t HoWo, float* dw, int cus, hipStream_t s) {
    return dy_f32 ? launch_bias<float>(dy, db, B, C, K, HoWo, dw, cus, s)
                  : launch_bias<_Float16>(dy, db, B, C, K, HoWo, dw, cus, s);
}

hipError_t launch_wgrad_direct(const uint16_t* x, const uint16_t* dy, float* dw, float* db, int B,
                               int C, int K, int H, int W, int pad, const WgradDirectPlan& p,
                               void* ws, hipStream_t s) {
    const int Ho = H + 2 * pad - 2, Wo = W + 2 * pad - 2;
    WdArgs a{};
    a.x = reinterpret_cast<const char*>(x);
    a.dy = reinterpret_cast<const char*>(dy);
    float* const part = static_cast<float*>(ws);
    float* const bpart = part + (int64_t)p.nsplit * 9 * K * C;
    a.out = p.nsplit > 1 ? part : dw;
    a.bias = db != nullptr && p.nsplit > 1 ? bpart : db;
    a.x_bytes = 2 * (int64_t)B * C * H * W;
    a.dy_bytes = 2 * (int64_t)B * K * Ho * Wo;
    a.B = B;
    a.C = C;
    a.K = K;
    a.H = H;
    a.W = W;
    a.Ho = Ho;
    a.Wo = Wo;
    a.G = p.G;
    a.R = p.R;
    a.nrb = p.nrb;
    a.Ws = p.Ws;
    a.nstrip = p.nstrip;
    a.lo = p.lo;
    a.XS = p.XS;
    a.XP = p.XP;
    a.xpitch = p.xpitch;
    a.dpitch = p.dpitch;
    a.dstart = p.dstart;
    a.zero = p.zero;
    a.nblk = p.nblk;
    a.nwx = p.nwx;
    a.mxp = (1u << 20) / (unsigned)p.xpitch + 1u;
    a.mdp = (1u << 20) / (unsigned)p.dpitch + 1u;
    a.mXP = magic(p.XP);
    a.mWs = magic(p.Ws);
    a.mR = magic(p.R);
    a.mR2 = magic(p.R + 2);
    a.ntk = p.ntk;
    a.nt = p.nt;
    a.nunits = p.nunits;
    a.nsplit = p.nsplit;
    a.nwg = p.nt * p.nsplit;
    // every row on a dword: straight to LDS
    const bool even = W % 2 == 0 && Wo % 2 == 0 && reinterpret_cast<uintptr_t>(x) % 4 == 0 &&
                      reinterpret_cast<uintptr_t>(dy) % 4 == 0;
    const int stage = !even ? kRegs : (W % 8 == 0 && Wo % 8 == 0) ? kDirect : kDirectTail;
    hipError_t e = pad == 0   ? launch_pad<0>(a, p, stage, s)
                   : pad == 1 ? launch_pad<1>(a, p, stage, s)
                              : launch_pad<2>(a, p, stage, s);
    if (e != hipSuccess || p.nsplit == 1) return e;
    const int64_t n = (int64_t)9 * K * C;
    const int nb = db != nullptr ? K : 0;
    launch(wgrad_direct_reduce_kernel,
           dim3((unsigned)((n + nb + kRedThreads - 1) / kRedThreads)), dim3(kRedThreads), s,
           static_cast<const float*>(part), dw, static_cast<const float*>(bpart), db, n, nb,
           p.nsplit);
    return hipGetLastError();
}

}  // namespace nova

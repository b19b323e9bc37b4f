// Winograd-domain batched GEMM on CDNA4 matrix cores (gfx950).
//
// Replaces the reference's rocBLAS call
// (/root/reference/csrc/nova_winograd.hip:589-601: 64 GEMMs, m=K, n=BP, k=C,
// fp16 operands, fp32 accumulate, fp16 result) with one hand-written kernel:
//
//   M_p[bp][k] = fp16( sum_c U_p[k][c] * V_p[bp][c] ),  p = 0..63
//
// Operand layouts keep the reduction index (c) contiguous so every lane feeds
// v_mfma_f32_16x16x32_f16 with one 16-byte load: A = U_p rows (16 k x 32 c),
// B = V_p rows (32 c x 16 bp). Lane l holds row/column (l % 16) and the eight
// channels 8*(l/16) .. 8*(l/16)+7 of the current 32-channel step; the
// accumulator lane holds D[4*(l/16) + i][l % 16]. The channel pitch Cp is a
// multiple of 8 and zero padded, so partial 32-channel steps only mask whole
// 8-channel groups. No atomics, no split-K: results are deterministic.
// Byte offsets are 32-bit: U, V and M must each stay below 2 GB.
#include <algorithm>
#include <type_traits>

#include "nova_internal.h"
#include "nova_tile_math.h"

namespace nova {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef unsigned int v2u __attribute__((ext_vector_type(2)));
typedef unsigned int v4u __attribute__((ext_vector_type(4)));

constexpr int kOob = (int)0x80000000;  // byte offset past every buffer: loads 0, stores dropped

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* p, int64_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0,
                                             (int)(bytes < 0x7fffffff ? bytes : 0x7fffffff),
                                             0x00020000);
}

// MT x NT 16x16 MFMA tiles per wave, WGM x WGN waves per workgroup. Operands
// are read through buffer resources: the per-lane part of each offset (row,
// channel octet) is fixed, the wave-uniform part (position, channel step)
// goes in a scalar offset, and lanes outside K / BP / Cp read zeros. A ring
// of PD channel steps is kept in flight (register prefetch) so the loop is
// not bound by load latency; steps past Cp are zero loads.
template <int MT, int NT, int WGM, int WGN, int PD>
__global__ __launch_bounds__(64 * WGM * WGN) void wgemm_kernel(
    const _Float16* __restrict__ U, const _Float16* __restrict__ V, _Float16* __restrict__ M,
    int K, int Cp, int BP) {
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int wm = wave % WGM, wn = wave / WGM;
    const int p = blockIdx.z;
    const int kbase = blockIdx.y * (MT * 16 * WGM) + wm * MT * 16;
    const int nbase = blockIdx.x * (NT * 16 * WGN) + wn * NT * 16;
    const int r16 = lane & 15;
    const int g = lane >> 4;

    const __amdgpu_buffer_rsrc_t urs = make_rsrc(U, 2 * (int64_t)64 * K * Cp);
    const __amdgpu_buffer_rsrc_t vrs = make_rsrc(V, 2 * (int64_t)64 * BP * Cp);
    const __amdgpu_buffer_rsrc_t mrs = make_rsrc(M, 2 * (int64_t)64 * BP * K);

    int aoff[MT], boff[NT];
#pragma unroll
    for (int mi = 0; mi < MT; mi++) {
        const int k = kbase + mi * 16 + r16;
        aoff[mi] = k < K ? 2 * (k * Cp + 8 * g) : kOob;
    }
#pragma unroll
    for (int ni = 0; ni < NT; ni++) {
        const int n = nbase + ni * 16 + r16;
        boff[ni] = n < BP ? 2 * (n * Cp + 8 * g) : kOob;
    }
    const int au = 2 * p * K * Cp;   // uniform
    const int bu = 2 * p * BP * Cp;  // uniform
    const int nsteps = (Cp + 31) / 32;

    h8 a[PD][MT], b[PD][NT];
    auto load_step = [&](int step, h8 af[MT], h8 bf[NT]) {
        const int c = step * 32;
        const bool cok = c + 8 * g < Cp;
#pragma unroll
        for (int mi = 0; mi < MT; mi++)
            af[mi] = __builtin_bit_cast(h8, __builtin_amdgcn_raw_buffer_load_b128(
                                                urs, cok ? aoff[mi] : kOob, au + 2 * c, 0));
#pragma unroll
        for (int ni = 0; ni < NT; ni++)
            bf[ni] = __builtin_bit_cast(h8, __builtin_amdgcn_raw_buffer_load_b128(
                                                vrs, cok ? boff[ni] : kOob, bu + 2 * c, 0));
    };

    f4 acc[MT][NT];
#pragma unroll
    for (int mi = 0; mi < MT; mi++)
#pragma unroll
        for (int ni = 0; ni < NT; ni++) acc[mi][ni] = f4{0.0f, 0.0f, 0.0f, 0.0f};

#pragma unroll
    for (int j = 0; j < PD; j++) load_step(j, a[j], b[j]);
    for (int s0 = 0; s0 < nsteps; s0 += PD) {
#pragma unroll
        for (int j = 0; j < PD; j++) {
#pragma unroll
            for (int mi = 0; mi < MT; mi++)
#pragma unroll
                for (int ni = 0; ni < NT; ni++)
                    acc[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[j][mi], b[j][ni],
                                                                         acc[mi][ni], 0, 0, 0);
            if (s0 + PD < nsteps) load_step(s0 + PD + j, a[j], b[j]);
        }
    }

    const int mu = 2 * p * BP * K;  // uniform
    const bool vec_store = (K & 3) == 0;
#pragma unroll
    for (int mi = 0; mi < MT; mi++)
#pragma unroll
        for (int ni = 0; ni < NT; ni++) {
            const int bp = nbase + ni * 16 + r16;
            const int k = kbase + mi * 16 + 4 * g;
            const int off = bp < BP ? 2 * (bp * K + k) : kOob;
            if (vec_store) {
                h4 v = {(_Float16)acc[mi][ni][0], (_Float16)acc[mi][ni][1],
                        (_Float16)acc[mi][ni][2], (_Float16)acc[mi][ni][3]};
                __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(v2u, v), mrs,
                                                      k < K ? off : kOob, mu, 0);
            } else {
#pragma unroll
                for (int i = 0; i < 4; i++)
                    __builtin_amdgcn_raw_buffer_store_b16(
                        __builtin_bit_cast(uint16_t, (_Float16)acc[mi][ni][i]), mrs,
                        k + i < K ? off + 2 * i : kOob, mu, 0);
            }
        }
}

template <int MT, int NT, int WGM, int WGN, int PD>
static hipError_t launch_cfg(const uint16_t* U, const uint16_t* V, uint16_t* M, int K, int Cp,
                             int BP, hipStream_t s) {
    constexpr int TM = MT * 16 * WGM, TN = NT * 16 * WGN;
    dim3 grid((unsigned)((BP + TN - 1) / TN), (unsigned)((K + TM - 1) / TM), 64);
    launch(wgemm_kernel<MT, NT, WGM, WGN, PD>, grid, dim3(64 * WGM * WGN), s,
        reinterpret_cast<const _Float16*>(U), reinterpret_cast<const _Float16*>(V),
        reinterpret_cast<_Float16*>(M), K, Cp, BP);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// LDS-tiled variant for larger shapes. Workgroup tile = TK output channels x
// TB tiles (bp) of one position, WK x WB waves, channels in stages of 64 (two
// MFMA k-steps, one 128-byte line per row when Cp >= 64). Stages go from
// memory to LDS directly (no registers in between), NST buffers, NST - 1
// stages ahead of the one that is multiplied. The buffers are separate arrays,
// each named by its own code: the compiler tells them apart and does not wait
// for a direct load into one before a read of another (with one array it
// waits for every load in flight, which is what made an earlier version of
// this slower than staging through registers).
//
// LDS rows are 128 bytes, 16-byte chunk c of row r at c ^ ((r >> 1) & 7):
// conflict-free on the 64 banks for the fragment reads (16 lanes on 16
// consecutive rows, one chunk each); a direct load writes 64 consecutive
// chunks, so its lanes fetch the permuted chunks of 8 rows' lines.
//
// What bounds it: L2 -> CU traffic, 2 * 64 * (nkt * BP + nbt * K) * Cp bytes
// (nkt, nbt: tiles along K and BP), at 7-10 TB/s, and the latency of a stage.
// Measured on MI355X (launch in a forward, us, 64-row tiles staged through
// registers -> this kernel with the rule's tile): 320@64^2 batch 16 62.6 ->
// 51.2 (64 x 128, 606 MB of traffic -> 160 x 128, 368 MB), batch 8 33.2 ->
// 27.2; 1280 -> 640@32^2 batch 2 32.4 -> 27.6; 1280@32^2 batch 4 78.8 -> 64.5;
// ResNet-50 batch 32 256@14^2 6.7 -> 6.2, 512@7^2 9.3 -> 8.9.
// ---------------------------------------------------------------------------
constexpr int kStageC = 64;

// A 16-byte store with a scalar offset. The data registers stay live over two
// wait states: written by the instruction right behind the store, they reach
// memory with the new value in the last lanes of each 16 (seen on gfx950; the
// compiler separates such pairs only for stores without a scalar offset).
__device__ __forceinline__ void store_b128(v4u v, __amdgpu_buffer_rsrc_t r, int off, int soff,
                                           bool write_through) {
    if (write_through)
        __builtin_amdgcn_raw_buffer_store_b128(v, r, off, soff, kWT);
    else
        __builtin_amdgcn_raw_buffer_store_b128(v, r, off, soff, 0);
    asm volatile("s_nop 1" ::"v"(v) : "memory");
}

template <int TK, int TB, int WK, int WB, int NST, int SM>
__global__ __launch_bounds__(64 * WK * WB) void wgemm_lds_kernel(const _Float16* __restrict__ U,
                                                        const _Float16* __restrict__ V,
                                                        _Float16* __restrict__ M, int K, int Cp,
                                                        int BP, int nwg) {
    constexpr int kWaves = WK * WB, kThreads = 64 * kWaves;
    constexpr int MT = TK / WK / 16;  // 16x16 tiles per wave along k
    constexpr int NT = TB / WB / 16;  // along bp
    constexpr int kBlkU = TK / 8, kBlkV = TB / 8;  // 1 KB blocks (8 rows) of a stage
    constexpr int kLoads = (kBlkU + kBlkV + kWaves - 1) / kWaves;  // per wave and stage
    constexpr int kBuf = kLoads * kWaves * 512;  // halves; blocks past the stage hold zeros
    __shared__ __align__(1024) _Float16 b0[kBuf];
    __shared__ __align__(1024) _Float16 b1[kBuf];
    __shared__ __align__(1024) _Float16 b2[NST > 2 ? kBuf : 8];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wk = wave % WK, wb = wave / WK;
    // One-dimensional grid, XCD-aware: every XCD takes a contiguous run of
    // (position, k-tile, bp-tile) items with the bp tile fastest, so all
    // tiles of a position meet in one L2 and U_p, V_p leave HBM once.
    const int nbt = (BP + TB - 1) / TB, nkt = (K + TK - 1) / TK;
    const int item = xcd_remap((int)blockIdx.x, nwg);
    const int p = item / (nbt * nkt);
    const int rem = item - p * (nbt * nkt);
    const int k0 = (rem / nbt) * TK;
    const int n0 = (rem % nbt) * TB;
    const int r16 = lane & 15, g = lane >> 4;

    const __amdgpu_buffer_rsrc_t urs = make_rsrc(U + (int64_t)p * K * Cp, 2 * (int64_t)K * Cp);
    const __amdgpu_buffer_rsrc_t vrs = make_rsrc(V + (int64_t)p * BP * Cp, 2 * (int64_t)BP * Cp);
    const __amdgpu_buffer_rsrc_t mrs = make_rsrc(M, 2 * (int64_t)64 * BP * K);

    // load j of the wave: block 8 rows x 8 chunks, lane = (row, slot)
    int off[kLoads], chan[kLoads];
#pragma unroll
    for (int j = 0; j < kLoads; j++) {
        const int blk = j * kWaves + wave;
        const bool u = blk < kBlkU;
        const int row = (u ? blk : blk - kBlkU) * 8 + (lane >> 3);
        chan[j] = 8 * ((lane & 7) ^ ((row >> 1) & 7));
        const int at = (u ? k0 : n0) + row;
        const bool ok = u ? at < K : blk < kBlkU + kBlkV && at < BP;
        off[j] = ok ? 2 * (at * Cp + chan[j]) : kOob;
    }
    const int nstages = (Cp + kStageC - 1) / kStageC;
    // stage st into buf; stages past the last one load zeros (NST > 2 counts
    // every stage's loads)
    auto issue = [&](int st, _Float16* buf) {
        const int c = st * kStageC;
#pragma unroll
        for (int j = 0; j < kLoads; j++) {
            const int blk = j * kWaves + wave;
            load_lds16(blk < kBlkU ? urs : vrs, buf + blk * 512,
                       c + chan[j] < Cp ? off[j] : kOob, 2 * c);
        }
    };

    f4 acc[MT][NT];
#pragma unroll
    for (int mi = 0; mi < MT; mi++)
#pragma unroll
        for (int ni = 0; ni < NT; ni++) acc[mi][ni] = f4{0.0f, 0.0f, 0.0f, 0.0f};
    // lane (row r16 of each 16-row tile, chunk 4*kk + g); every tile starts at
    // a multiple of 16 rows, so the swizzle depends on r16
    const int c0 = g ^ ((r16 >> 1) & 7);
    auto multiply = [&](const _Float16* buf) {
        const _Float16* su = buf + (wk * MT * 16 + r16) * kStageC;
        const _Float16* sv = buf + (TK + wb * NT * 16 + r16) * kStageC;
#pragma unroll
        for (int kk = 0; kk < kStageC / 32; kk++) {
            const int co = (c0 ^ (4 * kk)) * 8;
            h8 a[MT], b[NT];
#pragma unroll
            for (int ni = 0; ni < NT; ni++)
                b[ni] = *reinterpret_cast<const h8*>(sv + ni * 16 * kStageC + co);
#pragma unroll
            for (int mi = 0; mi < MT; mi++)
                a[mi] = *reinterpret_cast<const h8*>(su + mi * 16 * kStageC + co);
#pragma unroll
            for (int mi = 0; mi < MT; mi++)
#pragma unroll
                for (int ni = 0; ni < NT; ni++)
                    acc[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[mi], b[ni],
                                                                         acc[mi][ni], 0, 0, 0);
        }
    };
    // stage st's loads are over (the next NST - 2 stages' may be in flight);
    // the barrier also ends stage st - 1's products, whose buffer is loaded
    auto turn = [&](int st, const _Float16* cur, _Float16* next) {
        wait_vmcnt<kLoads * (NST - 2)>();
        lds_barrier();
        if (NST > 2 || st + 1 < nstages) issue(st + NST - 1, next);
        __builtin_amdgcn_sched_barrier(0);
        multiply(cur);
        __builtin_amdgcn_sched_barrier(0);
    };
    issue(0, b0);
    if constexpr (NST > 2) issue(1, b1);
    for (int st = 0; st < nstages; st += NST) {
        if constexpr (NST == 2) {
            turn(st, b0, b1);
            if (st + 1 < nstages) turn(st + 1, b1, b0);
        } else {
            turn(st, b0, b2);
            if (st + 1 < nstages) turn(st + 1, b1, b0);
            if (st + 2 < nstages) turn(st + 2, b2, b1);
        }
    }
    wait_vmcnt<0>();
    lds_barrier();

    const int mu = 2 * p * BP * K;
    // The M tile goes through LDS as [bp][k] rows, half of them in each
    // buffer, and leaves as whole rows, 16 bytes per lane (SM 2: written
    // through the L2, sc1); the L2 then holds whole lines instead of 32-byte
    // pieces of 16.
    if ((K & 7) == 0) {
        constexpr int kMP = TK + 8;    // halves per staged row
        constexpr int kRows = TB / 2;  // rows per buffer
        static_assert(kRows % 16 == 0 && kRows * kMP <= kBuf, "M tile fits in the stages");
#pragma unroll
        for (int mi = 0; mi < MT; mi++)
#pragma unroll
            for (int ni = 0; ni < NT; ni++) {
                const int bpl = (wb * NT + ni) * 16;  // uniform
                const int kl = (wk * MT + mi) * 16 + 4 * g;
                const h4 v = h4{(_Float16)acc[mi][ni][0], (_Float16)acc[mi][ni][1],
                                (_Float16)acc[mi][ni][2], (_Float16)acc[mi][ni][3]};
                if (bpl < kRows)
                    *reinterpret_cast<h4*>(b0 + (bpl + r16) * kMP + kl) = v;
                else
                    *reinterpret_cast<h4*>(b1 + (bpl - kRows + r16) * kMP + kl) = v;
            }
        lds_barrier();
        constexpr int kCh = TK / 8;  // 16-byte chunks per row
        auto rows_out = [&](const _Float16* buf, int bp0) {
#pragma unroll
            for (int e = tid; e < kRows * kCh; e += kThreads) {
                const int row = e / kCh, ch = e % kCh;
                const int bp = bp0 + row, k = k0 + 8 * ch;
                store_b128(*reinterpret_cast<const v4u*>(buf + row * kMP + 8 * ch), mrs,
                           (bp < BP && k < K) ? 2 * (bp * K + k) : kOob, mu, SM == 2);
            }
        };
        rows_out(b0, n0);
        rows_out(b1, n0 + kRows);
        return;
    }
    const bool vec_store = (K & 3) == 0;
#pragma unroll
    for (int mi = 0; mi < MT; mi++)
#pragma unroll
        for (int ni = 0; ni < NT; ni++) {
            const int bp = n0 + (wb * NT + ni) * 16 + r16;
            const int k = k0 + (wk * MT + mi) * 16 + 4 * g;
            const int off = bp < BP ? 2 * (bp * K + k) : kOob;
            if (vec_store) {
                h4 v = {(_Float16)acc[mi][ni][0], (_Float16)acc[mi][ni][1],
                        (_Float16)acc[mi][ni][2], (_Float16)acc[mi][ni][3]};
                __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(v2u, v), mrs,
                                                      k < K ? off : kOob, mu, 0);
            } else {
#pragma unroll
                for (int i = 0; i < 4; i++)
                    __builtin_amdgcn_raw_buffer_store_b16(
                        __builtin_bit_cast(uint16_t, (_Float16)acc[mi][ni][i]), mrs,
                        k + i < K ? off + 2 * i : kOob, mu, 0);
            }
        }
}

// M epilogue of the LDS kernels (SM of wgemm_lds_kernel): always staged
// through LDS as whole rows (K % 8 == 0); written through the L2 (sc1, so the
// launch boundary has no dirty M to write back before the output transform
// starts) when M holds at most 32 MB. Measured on MI355X, whole forwards, us
// (direct b64 stores -> staged): ResNet-50 batch 32 128@28^2 28.9 -> 28.0,
// 256@14^2 30.2 -> 29.6, 512@7^2 28.6 -> 27.1, conv2_x three-pass 40.8 ->
// 36.4; batch 128 128@28^2 70.3 -> 64.1; batch 1 64@56^2 10.9 -> 10.4.
// Staged, write-back -> written through (with the V of the input transform
// written through as well; GEMM + output transform launches, event-timed):
// batch 16 256@14^2 7.22 + 6.75 -> 6.42 + 5.95; batch 64 128@28^2 11.69 +
// 11.69 -> 10.54 + 11.56; SDXL 320@128^2 (20 MB) 13.86 + 11.36 -> 12.81 +
// 11.52; above 32 MB it loses (batch 128 512@7^2, 34 MB: 26.59 + 12.77 ->
// 28.06 + 15.25). Streaming M with nt instead (4-16 MB) gained 0.4-1.2 us.
static int m_epilogue(int K, int BP) {
    const int64_t m_bytes = 2 * (int64_t)64 * BP * K;
    return m_bytes <= ((int64_t)32 << 20) ? 2 : 1;
}

template <int TK, int TB, int WK, int WB, int NST>
static hipError_t launch_lds(const uint16_t* U, const uint16_t* V, uint16_t* M, int K, int Cp,
                             int BP, hipStream_t s) {
    const unsigned grid = 64u * (unsigned)((BP + TB - 1) / TB) * (unsigned)((K + TK - 1) / TK);
    auto go = [&](auto kernel) {
        launch_n(kernel, dim3(grid), dim3(64 * WK * WB), s, reinterpret_cast<const _Float16*>(U),
               reinterpret_cast<const _Float16*>(V), reinterpret_cast<_Float16*>(M), K, Cp, BP);
    };
    if (m_epilogue(K, BP) == 2)
        go(wgemm_lds_kernel<TK, TB, WK, WB, NST, 2>);
    else
        go(wgemm_lds_kernel<TK, TB, WK, WB, NST, 1>);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// GEMV-like shapes (BP <= 32, or 48 above K = 1024) on 1 KB operand blocks: U from the two-pass
// kernel's block copy (launch_u_wfrag: block (p, 16-row tile, 32-channel
// step), lane l = row l % 16, channels 8*(l / 16) .. +7) and V in the
// two-pass layout (launch_input_transform with vfrag = ceil(Cp / 32)), so
// every operand fragment is one contiguous 1 KB load per wave; the product
// layouts make it 16 rows x 64 bytes, two rows per 128-byte line with the
// line's other half fetched by the next step. Wave = MT 16-row tiles of K x
// all NT 16-tile blocks of BP; PD steps in flight; M leaves in the product
// layout [64][BP][K] for the output transform. Same lane layout and
// channel-step order as the other GEMM kernels: M is bit-identical. Measured
// on MI355X (back-to-back launches, us, product-layout kernel -> blocks):
// 512@7^2 batch 1 6.5 -> 4.6, batch 4 8.8 -> 4.7, batch 8 (32 tiles) 7.8 ->
// 6.5; 256@14^2 batch 1 3.1 -> 2.8, batch 3 4.1 -> 3.3; 128@28^2 batch 1 (25
// tiles) 3.1 -> 2.7; 1280@8^2 batch 1 33.4 -> 30.4, batch 2 35.1 -> 30.6 (U
// at 6.9 TB/s); 1280@16^2 batch 2 (18 tiles) 33.7 -> 31.3. Past 32 tiles
// (three blocks per wave) it won at 3 of 4 shapes (1280@32^2 batch 1, 36
// tiles, 35.2 -> 33.3; 512@7^2 batch 12 8.1 -> 7.3) and lost 7 % at 640@32^2
// batch 1, so it takes 33-48 tiles only above K = 1024 (whole forwards in a
// graph, us: 1280@32^2 batch 1 51.0 -> 49.0, 1280@36^2 51.7 -> 49.8; 1024@32^2
// batch 1 36.3 -> 36.5).
// ---------------------------------------------------------------------------
template <int MT, int NT, int PD, int WPB, int kPol>
__global__ __launch_bounds__(64 * WPB) void wgemm_block_kernel(
    const _Float16* __restrict__ Uw, const _Float16* __restrict__ Vb, _Float16* __restrict__ M,
    int K, int Cp, int BP, int u_bytes, int v_bytes, int m_bytes, int nwg) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int nkt = (K + 15) / 16;
    const int nkg = (nkt + MT - 1) / MT;
    // XCD-aware: each XCD takes a contiguous run of positions
    const int item = xcd_remap((int)blockIdx.x, nwg) * WPB + wave;
    if (item >= 64 * nkg) return;  // no barrier below: idle waves may leave
    const int p = item / nkg;
    const int kt0 = (item - p * nkg) * MT;
    const int nsteps = (Cp + 31) / 32;
    const int nbb = (BP + 15) / 16;  // <= NT
    const int r16 = lane & 15, g = lane >> 4;
    const __amdgpu_buffer_rsrc_t urs = make_rsrc(Uw, u_bytes);
    const __amdgpu_buffer_rsrc_t vrs = make_rsrc(Vb, v_bytes);
    const __amdgpu_buffer_rsrc_t mrs = make_rsrc(M, m_bytes);
    // U blocks hold zeros past K and Cp; V slots of tiles past BP and of
    // channels past Cp are never written, so those lanes read through
    // out-of-range offsets
    int aoff[MT], boff[NT];
#pragma unroll
    for (int i = 0; i < MT; i++)
        aoff[i] = kt0 + i < nkt ? (p * nkt + kt0 + i) * nsteps * 1024 + lane * 16 : kOob;
#pragma unroll
    for (int n = 0; n < NT; n++)
        boff[n] = 16 * n + r16 < BP ? ((p * nbb + n) * nsteps) * 1024 + lane * 16 : kOob;
    h8 a[PD][MT], b[PD][NT];
    auto load = [&](int j, h8 (&af)[MT], h8 (&bf)[NT]) {
        const bool cok = j < nsteps && 32 * j + 8 * g < Cp;  // Cp % 8 == 0: whole groups
#pragma unroll
        for (int i = 0; i < MT; i++)
            af[i] = __builtin_bit_cast(h8, __builtin_amdgcn_raw_buffer_load_b128(
                                               urs, j < nsteps ? aoff[i] : kOob, j * 1024, 0));
#pragma unroll
        for (int n = 0; n < NT; n++)
            bf[n] = __builtin_bit_cast(h8, __builtin_amdgcn_raw_buffer_load_b128(
                                               vrs, cok ? boff[n] : kOob, j * 1024, 0));
    };
    f4 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int n = 0; n < NT; n++) acc[i][n] = f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int j = 0; j < PD; j++) load(j, a[j], b[j]);
    for (int s0 = 0; s0 < nsteps; s0 += PD) {
#pragma unroll
        for (int j = 0; j < PD; j++) {
            if (s0 + j >= nsteps) break;
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int n = 0; n < NT; n++)
                    acc[i][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[j][i], b[j][n],
                                                                       acc[i][n], 0, 0, 0);
            if (s0 + PD + j < nsteps) load(s0 + PD + j, a[j], b[j]);
        }
    }
    const int mu = 2 * p * BP * K;  // uniform
    const bool vec_store = (K & 3) == 0;
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int n = 0; n < NT; n++) {
            const int k = (kt0 + i) * 16 + 4 * g;
            const int bp = 16 * n + r16;
            const int off = bp < BP ? 2 * (bp * K + k) : kOob;
            if (vec_store) {
                h4 v = {(_Float16)acc[i][n][0], (_Float16)acc[i][n][1], (_Float16)acc[i][n][2],
                        (_Float16)acc[i][n][3]};
                __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(v2u, v), mrs,
                                                      k < K ? off : kOob, mu, kPol);
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++)
                    __builtin_amdgcn_raw_buffer_store_b16(
                        __builtin_bit_cast(uint16_t, (_Float16)acc[i][n][e]), mrs,
                        k + e < K ? off + 2 * e : kOob, mu, kPol);
            }
        }
}

bool wgemm_blocks(int K, int Cp, int BP) {
    return (BP <= 32 || (BP <= 48 && K > 1024)) && 2 * u_frag_elems(K, Cp) < ((int64_t)1 << 31) &&
           2 * (int64_t)64 * BP * K < ((int64_t)1 << 31);
}

hipError_t launch_wgemm_blocks(const uint16_t* Uw, const uint16_t* Vb, uint16_t* M, int K,
                               int Cp, int BP, hipStream_t s) {
    if (!wgemm_blocks(K, Cp, BP) || Cp % 8 != 0) return hipErrorInvalidValue;
    if (BP == 0) return hipSuccess;
    constexpr int kMT = 2, kPD = 4, kWPB = 2;
    const int nkg = ((K + 15) / 16 + kMT - 1) / kMT;
    const unsigned grid = (unsigned)((64 * nkg + kWPB - 1) / kWPB);
    auto go = [&](auto kernel) {
        launch_n(kernel, dim3(grid), dim3(64 * kWPB), s, reinterpret_cast<const _Float16*>(Uw),
               reinterpret_cast<const _Float16*>(Vb), reinterpret_cast<_Float16*>(M), K, Cp, BP,
               (int)(2 * u_frag_elems(K, Cp)), (int)(2 * gemm_out_v_elems(Cp, BP)),
               (int)(2 * (int64_t)64 * BP * K));
    };
    // M (32-byte pieces of lines) written through the L2 while it is small
    // (batch-1 layers, kWTSmallBytes)
    const bool wt = 2 * (int64_t)64 * BP * K <= kWTSmallBytes;
    auto by_tiles = [&](auto pol) {
        constexpr int P = decltype(pol)::value;
        if (BP <= 16)
            go(wgemm_block_kernel<kMT, 1, kPD, kWPB, P>);
        else if (BP <= 32)
            go(wgemm_block_kernel<kMT, 2, kPD, kWPB, P>);
        else
            go(wgemm_block_kernel<kMT, 3, kPD, kWPB, P>);
    };
    if (wt)
        by_tiles(std::integral_constant<int, kWT>());
    else
        by_tiles(std::integral_constant<int, 0>());
    return hipGetLastError();
}

const char* wgemm_blocks_name(int BP) {
    return BP <= 16   ? "wgemm_block_kernel<2, 1, 4, 2>"
           : BP <= 32 ? "wgemm_block_kernel<2, 2, 4, 2>"
                      : "wgemm_block_kernel<2, 3, 4, 2>";
}

// Kernel per shape on the product layouts (the operand-block kernel above
// takes GEMV-like shapes when the handle can hold U's block copy; this rule
// serves the rest, and the allocation-free forward). Register-direct 64 x 16
// for GEMV-like batch-1 deep layers (BP <= 16: few tiles; two 16-row tiles
// per wave, which halves the V fragment loads and doubles the U bytes each
// wave keeps in flight: 512@7^2 at batch 1 7.1 -> 6.5 us, 1280@8^2 at batch
// 2 39.2 -> 34.9 us); LDS-tiled otherwise, the tile chosen from a sweep of
// every tile shape on MI355X (GEMM launches inside forwards, per-kernel
// events, us; the results are bit-identical across tile shapes). Tiles that
// leave no more of K empty than 64-row ones, as large as the work allows:
//  * 160 x 128 where 160 divides K as well as 64 does, from 240 tiles with a
//    workgroup for every CU (128 above K = 1024): fewer and larger workgroups read V and U less often
//    (320@64^2 B=16 60.3 for 64 x 128, 59.5 for 128 x 128, 51.0; B=8 33.4,
//    31.5, 27.4; 640@64^2 B=8 91.1, 81.8, 73.3; 160@28^2 B=32 13.1, 11.7,
//    10.4; 1280@32^2 B=4, 144 tiles, 76.5 for 64 x 96, 72.1, 66.6); below
//    that the grid is too small (640@64^2 B=1, 121 tiles: 14.6 against 13.6;
//    64 -> 160@24^2 B=16, 128 workgroups, a forward 17.1 against 16.2);
//  * the same tile with three buffers for deep layers at 64 to 128 tiles (U
//    streams from memory, one workgroup per CU: 1280 -> 640@32^2 B=2 27.6
//    against 30.2 with two buffers and 32.1 for 64 x 96; 640@64^2 B=1 12.3
//    against 13.6), below 1024 channels only where 96-tile widths do not fit
//    BP better (640@32^2 B=2, 72 tiles, 11.7 against 11.4; with 320 channels
//    8.7 against 7.6);
//  * 96 x 96 or 96 x 128 where 96 divides K as well, from 128 tiles (whole
//    forwards, eager, us: 384@20^2 B=12 24.9 for 64 x 64, 21.9; 480@30^2 B=6
//    31.9, 30.0; 192@28^2 B=32 34.4 for 64 x 128, 96 x 128 34.5, 96 x 96 33.5;
//    launch alone 96@56^2 B=16 12.7 for 64 x 128, 96 x 96 10.7, 96 x 128 9.7;
//    384@28^2 B=8 9.0, 9.5, 8.2), the width that fills BP better; up to K =
//    192 from 384 tiles, below which the grid is too small (whole forwards in a
//    graph: 480 -> 96@48^2 B=2 21.5 against 18.9 for 64 x 64, 96@14^2 B=16 12.5
//    and 11.7, 192@40^2 B=3 17.0 and 16.4); from K = 640 and 256 tiles, where
//    128 x 128 begins, only if 96 tiles fill BP 15 points better (768@56^2 B=4,
//    400 tiles, 100.3 against 87.7, 640 -> 768@64^2 B=4, 484, 99.8 and 91.2; 64 ->
//    768@14^2 B=32, 288 tiles, 23.0 and 24.1);
//  * 128 rows where 128 divides K as well: 128 x 192 from 500 tiles that it
//    fills (256@14^2 B=64 27.2 -> 26.4, B=128 54.0 -> 51.6 for whole
//    forwards), 128 x 128 from 300 (48 -> 200@21^2 B=20 19.0 -> 18.1), for
//    K >= 512 from 256 (512@7^2 B=64 13.9 vs 15.5-17.3 for the other shapes,
//    B=128 24.9 vs 26.2-30.8), for K of 97 to 128 from 1600 (128@28^2 B=64
//    10.7 for 64 x 128, 10.2, B=128 25.4, 22.8);
//  * 128 x 64 (8 waves) for K >= 1024 below 128 tiles (whole forwards, us,
//    against 64 x 64, 64 x 128 and 64 x 96: 1280@48^2 B=1 74.0 vs 78.2, 79.4,
//    78.9; 1280@32^2 B=2 77.7 vs 83.5, 80.9, 79.5; 1024@48^2 B=1 46.5 vs 48.0,
//    54.7, 49.0; up to 32 tiles, or 48 above K = 1024, the operand-block kernel
//    takes them). The three-buffer 160 x 128 tile, which stops below K = 1024, is
//    faster still where 160 divides K (67.8 and 69.1 at the first two) and
//    slower where it does not (51.0 at the third);
//  * 64 x 128 for larger work: K >= 640 from 64 tiles, K >= 512 from 128,
//    K >= 256 from 200 (512@7^2 B=32 9.0 vs 10.0 for 128 x 128; 256@14^2 B=24
//    18.7 vs 19.0);
//  * 64 x 96 with four waves where that tile width fills its last tile 15
//    points better than 128, for K >= 256 from 128 tiles (256@14^2 B=32, 288
//    tiles, 6.6 against 7.5, B=16 16.3 -> 15.9 for a forward; 640@32^2 B=2, 72
//    tiles, 11.4 against 12.4);
//  * else 64 x 64: four waves from 300 workgroups, eight below (210 layers that
//    the rules above leave: up to 300 eight take 2 % of a forward less, at 300 to
//    400 they are equal, above that four take 1-4 % less); off 4, where M is
//    stored value by value, eight up to K = 256 (14 layers: 1 % less on average,
//    500 -> 189@40^2 B=4 31.4 against 32.4) and four above. Channel counts off 8
//    (M stored in pieces) have only the rules without fill: 64 rows (189@15^2
//    B=45 28.5 against 30.0 for 96 x 128), and the 128-row tiles of K >= 512 from
//    256 tiles and K >= 1024 below 128 (517@33^2 B=9 45.9 against 44.2 for 64
//    rows, 1029@33^2 B=16 119.9 against 119.0-122.6, 1030@25^2 B=2 45.4 against
//    45.7-48.5).
// Share of a row of tiles of width t that n fills.
static double fill(int n, int t) { return (double)n / (t * ((n + t - 1) / t)); }

static int wgemm_cfg(int K, int Cp, int BP) {
    if (BP <= 16) return 0;
    const bool narrow = fill(BP, 96) >= fill(BP, 128) + 0.15;
    const auto grid = [=](int tk, int tb) {  // workgroups
        return (int64_t)64 * ((K + tk - 1) / tk) * ((BP + tb - 1) / tb);
    };
    if (K % 8 == 0) {
        if (K >= 160 && fill(K, 160) >= fill(K, 64)) {
            if ((BP >= 240 && grid(160, 128) >= 256) || (K >= 1024 && BP >= 128)) return 8;
            if (K >= 640 && K < 1024 && Cp >= (narrow ? 1024 : 640) && BP >= 64 && BP <= 128)
                return 9;
        }
        if (BP >= 128 && K >= 65 && fill(K, 96) >= std::max(fill(K, 64), fill(K, 128)) &&
            (K > 192 || BP >= 384) && (K < 640 || BP < 256 || narrow))
            return fill(BP, 96) >= fill(BP, 128) + 0.03 ? 11 : 10;
        if (K >= 192 && fill(K, 128) >= fill(K, 64)) {
            if (BP >= 500 && fill(BP, 192) >= fill(BP, 128)) return 3;
            if (BP >= 300) return 2;
        }
        if (BP >= 1600 && K > 96 && K <= 128) return 2;
    }
    if (K >= 512 && BP >= 256) return 2;
    if (K >= 1024 && BP < 128) return 5;
    if (K >= 256 && BP >= 128 && narrow) return 7;
    if ((K >= 640 && BP >= 64) || (K >= 512 && BP >= 128) || (K >= 256 && BP >= 200) ||
        (K <= 128 && BP >= 1600))
        return narrow ? 7 : 6;
    return (K % 4 == 0 ? grid(64, 64) >= 300 : K > 256) ? 1 : 4;
}

int wgemm_stream_v(int K, int Cp, int BP) {
    static const int tk[] = {64, 64, 128, 128, 64, 128, 64, 64, 160, 160, 96, 96};
    const int cfg = wgemm_cfg(K, Cp, BP);
    const int64_t v_bytes = 2 * (int64_t)64 * Cp * BP, m_bytes = 2 * (int64_t)64 * K * BP;
    if (cfg == 9 && 2 * (int64_t)64 * K * Cp >= ((int64_t)96 << 20)) return 2;
    if (v_bytes > ((int64_t)24 << 20) || (K + tk[cfg] - 1) / tk[cfg] > 4) return 0;
    if (K <= 256 || (K == 512 && BP >= 256)) return 1;
    return Cp % 32 == 0 && (v_bytes >= ((int64_t)12 << 20) || m_bytes >= ((int64_t)32 << 20));
}

const char* wgemm_name(int K, int Cp, int BP) {
    static const char* names[] = {"wgemm_kernel<2, 1, 2, 1, 4>", "wgemm_lds_kernel<64, 64, 2, 2, 2>",
                                  "wgemm_lds_kernel<128, 128, 2, 4, 2>",
                                  "wgemm_lds_kernel<128, 192, 2, 4, 2>",
                                  "wgemm_lds_kernel<64, 64, 2, 4, 2>",
                                  "wgemm_lds_kernel<128, 64, 2, 4, 2>",
                                  "wgemm_lds_kernel<64, 128, 2, 4, 2>",
                                  "wgemm_lds_kernel<64, 96, 2, 2, 2>",
                                  "wgemm_lds_kernel<160, 128, 2, 4, 2>",
                                  "wgemm_lds_kernel<160, 128, 2, 4, 3>",
                                  "wgemm_lds_kernel<96, 128, 2, 4, 2>",
                                  "wgemm_lds_kernel<96, 96, 2, 2, 2>"};
    return names[wgemm_cfg(K, Cp, BP)];
}

hipError_t launch_wgemm(const uint16_t* U, const uint16_t* V, uint16_t* M, int K, int Cp,
                        int BP, hipStream_t s) {
    switch (wgemm_cfg(K, Cp, BP)) {
        case 0: return launch_cfg<2, 1, 2, 1, 4>(U, V, M, K, Cp, BP, s);
        case 1: return launch_lds<64, 64, 2, 2, 2>(U, V, M, K, Cp, BP, s);
        case 2: return launch_lds<128, 128, 2, 4, 2>(U, V, M, K, Cp, BP, s);
        case 3: return launch_lds<128, 192, 2, 4, 2>(U, V, M, K, Cp, BP, s);
        case 5: return launch_lds<128, 64, 2, 4, 2>(U, V, M, K, Cp, BP, s);
        case 6: return launch_lds<64, 128, 2, 4, 2>(U, V, M, K, Cp, BP, s);
        case 7: return launch_lds<64, 96, 2, 2, 2>(U, V, M, K, Cp, BP, s);
        case 8: return launch_lds<160, 128, 2, 4, 2>(U, V, M, K, Cp, BP, s);
        case 9: return launch_lds<160, 128, 2, 4, 3>(U, V, M, K, Cp, BP, s);
        case 10: return launch_lds<96, 128, 2, 4, 2>(U, V, M, K, Cp, BP, s);
        case 11: return launch_lds<96, 96, 2, 2, 2>(U, V, M, K, Cp, BP, s);
        default: return launch_lds<64, 64, 2, 4, 2>(U, V, M, K, Cp, BP, s);
    }
}

}  // namespace nova

// Slab-resident BF16 GEMM for gfx950 at K = 384 (the Julia-1 shape's Wqkv, Wo
// and Wi, and its head's K = 384 projections).
//
// out = epi(X · Wᵀ) as in gemm.hip.  A workgroup of NW waves keeps a slab of
// 32·NW rows of W in registers (wave w: two 16-row groups "lo" and "hi" of the
// slab's 64-row block w / 2, 96 VGPRs) and multiplies it with a range of tokens,
// which arrive by DMA in units of 16 through a ring in LDS.  NW = 4: 128-row
// slabs, two workgroups per CU, for outputs of a few hundred tokens up; NW = 12:
// 384-row slabs, one per CU, which read X a third as often, for large batches.
//
// Why: at K = 384 a 128x128 tile has only six K steps, so the tiled kernels
// spend most of a launch on the latency of each step's DMA and re-read W per
// tile, and the small-batch kernel re-reads W for every 32 tokens.  Here all of a
// workgroup's W and its first units of X are in flight at once, and neither is
// fetched again.  What is left at a few thousand tokens is the launch, the first
// fetch of W (60 B/ns per CU while every CU fetches) and the last stores; at
// 65536 tokens the output and X through HBM (N = 1152: 201 MB, 40 us of 66).
//
// The 16x16x32 accumulators leave lane (tk, kg) with token tk and rows 4kg ..
// +3 of each group; rows 16(w % 2) and 32 + 16(w % 2) of a 64-row block are
// the RoPE pair (d, d + 32) and the GEGLU pair (gate, up).  For the FP32
// outputs the operands change places (the same products in the same order):
// lane (tk, kg) then holds row tk of each group and tokens 4kg .. +3, and
// adjacent lanes load and store adjacent columns.  bf16 outputs go through LDS
// to whole-row stores: 8-byte stores of 16 tokens side by side ran at 19 B/ns
// per CU in a probe, against 55 along rows.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "../../include/julia1_hip_ops.h"
#include "kernels.hpp"

namespace {

constexpr int SL_K = 384;
constexpr int SL_KJ = SL_K / 64;         // 128-byte row segments
constexpr int SL_UNIT = 16;              // tokens per ring slot
constexpr int SL_X = SL_UNIT * SL_K;     // bf16 elements of X per unit (12 KB)
constexpr int SL_CS = 2 * SL_UNIT * 32;  // floats of a unit's cos and sin rows (4 KB)

typedef const __attribute__((address_space(4))) int32_t const_i32;

__device__ constexpr int swz(int r) { return (r >> 1) & 7; }

// s_waitcnt vmcnt: all but this wave's N most recent vector-memory operations
// have completed (63 is the most that the counter holds).
template <int N>
__device__ inline void wait_vm() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N < 63 ? N : 63) : "memory");
}

template <int EPI, int NW>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(NW == 4 ? 2 : 3))) void gemm_slab_kernel(
    GemmArgs a, int nF, int R, int nU) {
    constexpr int SL_ROWS = 32 * NW;     // W rows per workgroup
    constexpr int SL_SW = NW * 4096;     // bytes: 4 KB per wave for W on its way to registers
    constexpr bool ROPE = EPI == JH_EPI_ROPE_BF16;
    constexpr bool GEGLU = EPI == JH_EPI_GEGLU_BF16;
    constexpr bool RESID = EPI == JH_EPI_RESID_F32;
    constexpr bool F32OUT = RESID || EPI == JH_EPI_BIAS_F32;
    constexpr bool BIASED = EPI == JH_EPI_BIAS_BF16 || EPI == JH_EPI_BIAS_RELU_BF16 || EPI == JH_EPI_BIAS_F32;
    constexpr int NU = NW == 4 ? 4 : ROPE ? 6 : 8;           // ring slots (48 or 64 KB; 96 KB)
    constexpr int XI = 12 / NW;                              // X DMA instructions per wave and unit
    constexpr int NX = XI + (ROPE && NW == 4 ? 1 : 0);       // all DMA of a wave and unit, at least
    constexpr int SLOT = SL_X * 2 + (ROPE ? SL_CS * 4 : 0);  // bytes
    // bf16 outputs of a unit on their way to whole-row stores: [token][column],
    // 16-byte chunks XOR-swizzled by the token so that the accumulators' 8-byte
    // writes (16 tokens side by side) spread over all banks.
    constexpr int OW = GEGLU ? SL_ROWS / 2 : SL_ROWS, OUNIT = SL_UNIT * OW * 2;
    constexpr int STAGE = F32OUT ? SL_SW : std::max(SL_SW, 4 * OUNIT);  // two steps of two units
    auto oswz = [](int t) { return GEGLU ? (t >> 1) & 7 : t; };
    // Vector-memory operations of a wave per step besides its two refill DMAs.
    constexpr int PER = F32OUT ? (RESID ? 32 : 16) : (GEGLU ? 1 : 2);
    __shared__ __align__(1024) uint8_t ring[NU * SLOT];
    __shared__ __align__(1024) uint8_t stage[STAGE];
    auto slot_x = [&](int k) { return (bf16_t*)&ring[(k % NU) * SLOT]; };
    auto slot_cs = [&](int k) { return (float*)&ring[(k % NU) * SLOT + SL_X * 2]; };

    const int lane = threadIdx.x & 63, tk = lane & 15, kg = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // Workgroup -> (token range r, slab f): consecutive u share r, and an XCD
    // (workgroup b runs on XCD b % 8) takes a contiguous run of u.
    const int G = gridDim.x, bid = blockIdx.x;
    const int xcd = bid & 7, q8 = G >> 3, r8 = G & 7;
    const int u = xcd * q8 + (xcd < r8 ? xcd : r8) + (bid >> 3);
    const int r = u / nF, f = u - r * nF;
    const int u0 = (int)((long)r * nU / R), nu = (int)((long)(r + 1) * nU / R) - u0;  // this range's units
    if (nu <= 0) return;

    // DMA of unit k into its slot: 12 instructions of [8 rows][128 B], one per
    // wave: rows 8(w % 2) .. +7 of segment w / 2; lane i takes row i / 8 and the
    // 16-byte chunk that belongs in slot i % 8.  Rows past the last token, and
    // units past the range, read zeros into slots that nothing is stored from.
    // With RoPE, waves 0-3 also bring the unit's cos and sin rows.
    const int drow = 8 * (wave & 1) + (lane >> 3);
    const uint32_t dchunk = (uint32_t)(((lane & 7) ^ swz(drow)) * 16);
    const uint32_t xoff = (uint32_t)drow * (uint32_t)a.ldx * 2 + dchunk;
    const bool rot_slab = ROPE && SL_ROWS * f < a.rope_cols;
    auto issue = [&](int k) {
        const int t0 = (u0 + k) * SL_UNIT;
        const i32x4 rx = k < nu ? make_rsrc(a.x + (long)t0 * a.ldx,
                                            (uint64_t)(a.rows - 1 - t0) * a.ldx * 2 + (uint64_t)SL_K * 2)
                                : make_rsrc(a.x, 0);
#pragma unroll
        for (int j = 0; j < XI; ++j) {
            const int seg = (wave >> 1) + j * (NW / 2);
            const uint32_t m0 =
                __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)slot_x(k) + seg * 2048 + (wave & 1) * 1024);
            asm volatile("buffer_load_dwordx4 %1, %2, %3 offen lds" ::"{m0}"(m0), "v"(xoff), "s"(rx), "s"(seg * 128)
                         : "memory");
        }
        if constexpr (ROPE) {
            if (wave < 4) {
                // The wave's eight positions, by scalar loads (a vector load's
                // wait would also wait for the DMA issued before it).
                uint32_t p = 0;
                if (rot_slab && k < nu) {
                    const_i32* pos = (const_i32*)a.pos;
                    const int first = t0 + 8 * (wave & 1);
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        const uint32_t pi = (uint32_t)pos[std::min(first + i, a.rows - 1)] & 0xffffu;
                        p = (lane >> 3) == i ? pi : p;
                    }
                }
                const i32x4 rt = make_rsrc((wave & 2) ? a.sin_t : a.cos_t, rot_slab && k < nu ? 65536ull * 128 : 0);
                const uint32_t mc = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)slot_cs(k) + wave * 1024);
                asm volatile("buffer_load_dwordx4 %1, %2, %3 offen lds" ::"{m0}"(mc), "v"(p * 128 + dchunk), "s"(rt),
                             "s"(0)
                             : "memory");
            }
        }
    };
    const int hb = SL_ROWS / 64 * f + (wave >> 1), x0 = 16 * (wave & 1);  // 64-row block of W, first row of "lo" in it

    // Output resource of unit k: it ends at the unit's last token, so that rows
    // past it are dropped (or read as 0).
    constexpr int ESZ = F32OUT ? 4 : 2;
    auto out_rsrc = [&](int k) {
        const int t0 = (u0 + k) * SL_UNIT, nt = std::min(a.rows - t0, SL_UNIT);
        return __builtin_amdgcn_make_buffer_rsrc((char*)a.out + (long)t0 * a.ldo * ESZ, 0,
                                                 k < nu ? (int)(nt * a.ldo * ESZ) : 0, 0x00020000);
    };

    // Bias of this lane's columns, loaded ahead of everything that is waited for later.
    f32x4 bias[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        bias[h] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        if ((BIASED || RESID) && a.bias) {
            if constexpr (F32OUT) bias[h][0] = a.bias[64 * hb + x0 + 32 * h + tk];
            else bias[h] = *(const f32x4*)(a.bias + 64 * hb + x0 + 32 * h + 4 * kg);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    issue(0);
    issue(1);
    // W: whole 128-byte row segments, eight rows per load, so that adjacent
    // lanes read adjacent memory (loads in the fragments' own lane order, 16
    // rows side by side, ran at 36 instead of 120 B/ns per CU in a probe).  Each
    // wave turns its rows into fragments through 4 KB of LDS of its own.
    u32x4 wr[SL_KJ][4];
    const bf16_t* wp = a.w + (long)(64 * hb + x0 + (lane >> 3)) * SL_K + (lane & 7) * 8;
#pragma unroll
    for (int j = 0; j < SL_KJ; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) wr[j][i] = *(const u32x4*)(wp + ((i >> 1) * 32 + (i & 1) * 8) * SL_K + j * 64);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 2; k < NU; ++k) issue(k);
    bf16x8 wf[2 * SL_KJ][2];
    bf16_t* const sw = (bf16_t*)stage + wave * 2048;
#pragma unroll
    for (int j = 0; j < SL_KJ; ++j) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int row = 8 * i + (lane >> 3);  // 0 .. 15 lo, 16 .. 31 hi
            *(u32x4*)&sw[row * 64 + (((lane & 7) ^ swz(row)) * 8)] = wr[j][i];
        }
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int row = 16 * h + tk;
                wf[2 * j + e][h] = *(const bf16x8*)&sw[row * 64 + (((4 * e + kg) ^ swz(row)) * 8)];
            }
    }

    // bf16 outputs: wave w stores 1 KB of each unit (of one of the two, GEGLU), 16
    // bytes per lane along the rows.
    constexpr int CPR = OW / 8, WPU = OUNIT / 1024;  // 16-byte chunks per output row; waves that store a unit
    const int oi = (wave % WPU) * 64 + lane, otok = oi / CPR, och = oi - otok * CPR;
    auto store_out = [&](int st) {
        if constexpr (!F32OUT) {
#pragma unroll
            for (int v = 0; v < (GEGLU ? 1 : 2); ++v) {
                const int un = GEGLU ? wave / WPU : v;
                const u32x4 d = *(const u32x4*)&stage[((st & 1) * 2 + un) * OUNIT + otok * OW * 2 + (och ^ oswz(otok)) * 16];
                __builtin_amdgcn_raw_buffer_store_b128(d, out_rsrc(2 * st + un),
                                                       (int)(otok * a.ldo + a.col + OW * f + och * 8) * 2, 0, 0);
            }
        }
    };

    const int nst = (nu + 1) >> 1;
    for (int st = 0; st < nst; ++st) {
        // This step's units (2st and 2st + 1) have landed for every wave and
        // the slots of the step before are free.  The counts are the operations
        // issued after those units' DMA, at least: the prologue's later units,
        // the refills of the steps since (one step's before the ring has gone
        // round), and what those steps load and store besides.
        constexpr int D = NU / 2, S0 = F32OUT ? PER : 0;  // S0: step 0 stores already (nothing is staged)
        if (st == 0) wait_vm<(NU - 2) * NX>();
        else if (st == 1) wait_vm<(NU - 4) * NX + S0>();
        else if (D > 2 && st == 2) wait_vm<(NU - 6) * NX + S0 + 2 * NX + PER>();
        else if (st < D) wait_vm<(NU - 8) * NX + S0 + 2 * (2 * NX + PER)>();
        else wait_vm<PER + (D - 2) * (2 * NX + PER)>();
        __syncthreads();
        if (st > 0) {
            issue(2 * st - 2 + NU);
            issue(2 * st - 1 + NU);
            store_out(st - 1);
        }
        // RESID: lane (tk, kg) adds to columns tk of each group of tokens 4kg ..
        // +3; adjacent lanes take adjacent columns.
        const int fcol = a.col + 64 * hb + x0 + tk;
        float old[2][2][4];
        if constexpr (RESID)
#pragma unroll
            for (int v = 0; v < 2; ++v) {
                const __amdgpu_buffer_rsrc_t ro = out_rsrc(2 * st + v);
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        old[v][h][i] = __builtin_bit_cast(
                            float, __builtin_amdgcn_raw_buffer_load_b32(
                                       ro, (int)((4 * kg + i) * a.ldo + fcol + 32 * h) * 4, 0, 0));
            }
        auto rd = [&](int s, int v) {
            return *(const bf16x8*)&slot_x(2 * st + v)[(s >> 1) * 1024 + tk * 64 + (((4 * (s & 1) + kg) ^ swz(tk)) * 8)];
        };
        f32x4 acc[2][2];  // [unit][lo/hi]
#pragma unroll
        for (int v = 0; v < 2; ++v)
#pragma unroll
            for (int h = 0; h < 2; ++h) acc[v][h] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        // 48 MFMAs, four per 32-deep K slice, with fragment reads PD slices ahead.
        constexpr int PD = RESID ? 2 : 3;
        bf16x8 bx[PD][2];
#pragma unroll
        for (int p = 0; p < PD; ++p)
#pragma unroll
            for (int v = 0; v < 2; ++v) bx[p][v] = rd(p, v);
#pragma unroll
        for (int s = 0; s < 2 * SL_KJ; ++s) {
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int v = 0; v < 2; ++v)
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    acc[v][h] = F32OUT ? __builtin_amdgcn_mfma_f32_16x16x32_bf16(bx[s % PD][v], wf[s][h], acc[v][h], 0, 0, 0)
                                       : __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[s][h], bx[s % PD][v], acc[v][h], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            if (s + PD < 2 * SL_KJ)
#pragma unroll
                for (int v = 0; v < 2; ++v) bx[s % PD][v] = rd(s + PD, v);
        }
#pragma unroll
        for (int v = 0; v < 2; ++v) {
            f32x4 lo = acc[v][0], hi = acc[v][1];
            if constexpr (ROPE) {
                if (hb * 64 < a.rope_cols) {
                    const float* C = slot_cs(2 * st + v) + tk * 32 + ((((x0 >> 2) + kg) ^ swz(tk)) * 4);
                    const f32x4 c = *(const f32x4*)C, sn = *(const f32x4*)(C + SL_UNIT * 32);
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        float l = lo[i], h = hi[i];
                        rope_rotate(l, h, c[i], sn[i]);
                        lo[i] = l;
                        hi[i] = h;
                    }
                }
            }
            if constexpr (GEGLU) {
#pragma unroll
                for (int i = 0; i < 4; ++i) lo[i] = gelu_erf(lo[i]) * hi[i];
            }
            if constexpr (BIASED || RESID) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (BIASED || a.bias) {
                        lo[i] += bias[0][F32OUT ? 0 : i];
                        hi[i] += bias[1][F32OUT ? 0 : i];
                    }
                    if constexpr (EPI == JH_EPI_BIAS_RELU_BF16) {
                        lo[i] = fmaxf(lo[i], 0.0f);
                        hi[i] = fmaxf(hi[i], 0.0f);
                    }
                    if constexpr (RESID) {
                        lo[i] = old[v][0][i] + lo[i];
                        hi[i] = old[v][1][i] + hi[i];
                    }
                }
            }
            if constexpr (F32OUT) {
                const __amdgpu_buffer_rsrc_t ro = out_rsrc(2 * st + v);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int vo = (int)((4 * kg + i) * a.ldo + fcol) * 4;
                    // (a scalar first: the compiler reads element 0 for a bit_cast of any vector element)
                    const float l = lo[i], h = hi[i];
                    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, l), ro, vo, 0, 0);
                    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, h), ro, vo + 128, 0, 0);
                }
            } else {
                // columns of the slab: 64 (32, GEGLU) per block of W, this lane's four in each half
                uint8_t* const d = &stage[((st & 1) * 2 + v) * OUNIT + tk * OW * 2];
                auto at = [&](int c) { return d + (((c >> 3) ^ oswz(tk)) * 16) + (c & 4) * 2; };
                const int c0 = (GEGLU ? 32 : 64) * (wave >> 1) + x0 + 4 * kg;
                *(u32x2*)at(c0) = u32x2{pack2(lo[0], lo[1]), pack2(lo[2], lo[3])};
                if constexpr (!GEGLU) *(u32x2*)at(c0 + 32) = u32x2{pack2(hi[0], hi[1]), pack2(hi[2], hi[3])};
            }
        }
    }
    if constexpr (!F32OUT) {
        __syncthreads();
        store_out(nst - 1);
    }
}

}  // namespace

bool gemm_slab_supported(int epi, const GemmArgs& a) {
    return a.k == SL_K && a.n % 128 == 0 && !a.gather && !a.xf && a.rows > 0 && a.w && gemm_offsets_fit(epi, a);
}

namespace {

template <int NW>
void launch_slab(int epi, const GemmArgs& a, int nF, int R, int nU, hipStream_t s) {
    const dim3 grid((unsigned)(nF * R)), block(64 * NW);
    switch (epi) {
        case JH_EPI_STORE_BF16: JH_LAUNCH((gemm_slab_kernel<JH_EPI_STORE_BF16, NW>), grid, block, 0, s, a, nF, R, nU); break;
        case JH_EPI_ROPE_BF16: JH_LAUNCH((gemm_slab_kernel<JH_EPI_ROPE_BF16, NW>), grid, block, 0, s, a, nF, R, nU); break;
        case JH_EPI_GEGLU_BF16: JH_LAUNCH((gemm_slab_kernel<JH_EPI_GEGLU_BF16, NW>), grid, block, 0, s, a, nF, R, nU); break;
        case JH_EPI_RESID_F32: JH_LAUNCH((gemm_slab_kernel<JH_EPI_RESID_F32, NW>), grid, block, 0, s, a, nF, R, nU); break;
        case JH_EPI_BIAS_BF16: JH_LAUNCH((gemm_slab_kernel<JH_EPI_BIAS_BF16, NW>), grid, block, 0, s, a, nF, R, nU); break;
        case JH_EPI_BIAS_RELU_BF16:
            JH_LAUNCH((gemm_slab_kernel<JH_EPI_BIAS_RELU_BF16, NW>), grid, block, 0, s, a, nF, R, nU);
            break;
        case JH_EPI_BIAS_F32: JH_LAUNCH((gemm_slab_kernel<JH_EPI_BIAS_F32, NW>), grid, block, 0, s, a, nF, R, nU); break;
        default: throw jh_error(1, "gemm: unknown epilogue");
    }
    HIP_CHECK(hipGetLastError());
}

}  // namespace

void launch_gemm_slab(int epi, const GemmArgs& a, int waves, hipStream_t s) {
    if (!gemm_slab_supported(epi, a) || (waves != 4 && (waves != 12 || a.n % 384)))
        throw jh_error(1, "gemm: the slab kernel needs K = 384 and N a multiple of its 128 or 384 rows, and rows of X "
                          "and the output under 2^28 bytes");
    // Token ranges per slab: as many as give two workgroups of four waves, or one
    // of twelve, per CU; at least one unit each.
    const int nU = (a.rows + SL_UNIT - 1) / SL_UNIT, slots = gemm_resident_tiles() / (waves == 4 ? 1 : 2);
    const int nF = a.n / (32 * waves), R = std::max(1, std::min(nU, slots / nF));
    if (waves == 12) launch_slab<12>(epi, a, nF, R, nU, s);
    else launch_slab<4>(epi, a, nF, R, nU, s);
}

// fp32 fused cross-attention for 16-latent workgroups on fp32 MFMA
// (v_mfma_f32_16x16x4_f32), gfx950: the form for batches and latent counts
// that 64-latent workgroups would leave the device half empty on, over longer
// key ranges (launch_flash_f32 has the rule).
//
// Work item = (batch b, key split s, block of 16 latents) on 4 wavefronts;
// wavefront w owns columns 192 w .. 192 w + 191 of Q, K, V and O.  Per 16-key
// tile it computes its columns' share of S^T[16 keys x 16 q] (48 MFMAs), the
// four shares meet in LDS, every wavefront adds them in the same order and
// takes the tile's weights (the passes of xattn_flash_f32.hip), and
// O[16 q x 192] += P . V[16 x 192] (48 MFMAs).  Computing S^T leaves the
// weights in the layout of the P operand.
//
// What bounds it: the MFMA pipe, 3,072 cycles per tile and SIMD, and beside
// an fp32 MFMA stream vector instructions are not hidden (one between two
// MFMAs costs 13 cycles, each further one 4; LDS reads, loads to registers and
// DMA cost nothing).  So:
//   * no wavefront reads another's columns, so tiles need no barrier: K comes
//     by DMA into the wavefront's own ring of three LDS slices, V by loads
//     straight into the operand's registers (its lanes lie on consecutive
//     bytes).  V(t) is requested a whole tile before its MFMAs.  K(t + 2) is
//     requested one and a half tiles before its first read, but has about half
//     a tile to arrive: the compiler, which counts the V loads and not the
//     DMA, waits before each output group for vmcnt(11), and the counter is in
//     order, so group n of V(t - 1) also waits for piece n of K(t + 2),
//     requested 48 MFMAs earlier;
//   * tile t's scores come before tile t - 1's output product, so the one
//     barrier of a tile and the exchange's reads pass under MFMAs (the write
//     of the shares does not: it waits for the last score MFMA's result);
//   * the tile loop is unrolled over the three slices, so LDS addresses are
//     registers set up once plus immediates, and the softmax is one run of
//     vector instructions per tile.
// Per tile 1.46 us with 64 workgroups (3,490 cycles at 2.40 GHz) and 1.49-1.51
// with 256, in the same cycles at the lower clock of a full device, against
// 1.59 and 1.61 us of the column-split form of flash_f32_kernel, whose
// wavefronts share row-wise tiles through two barriers per tile.  B=8 NL=512
// NI=784: 79.0 against 84.4 us per call.  Measured and not kept: a tile's
// weights dealt to the four wavefronts (a quarter of the vector instructions,
// one more exchange: the same time); K through registers and ds_write
// (1.86 us per tile: ds_write_b128 moves 76 B/clk per CU); the loop not
// unrolled (3 % slower at 49 tiles); DMA chunks in the operands' order (64
// bytes of 16 rows each: 3 % slower, 10 % with inputs from HBM); V two tiles
// ahead (the same).
#include "xattn_common.h"
#include "xattn_launch.h"

namespace xattn {
namespace f32s {

constexpr int BN = 16;                 // keys per tile
constexpr int BM = 16;                 // latents per workgroup
constexpr int NW = 4;                  // wavefronts per workgroup, one per SIMD
constexpr int DW = kDim / NW;          // columns of Q, K, V and O per wavefront (192)
constexpr int NU = DW / 16;            // K operands per tile and wavefront (12)
constexpr int NT = DW / 64;            // 64-column output blocks per wavefront (3)
constexpr int NCH = BN * DW / 4 / kWave;  // 1 KiB loads per wavefront's tile slice (12)
constexpr int ROWB = kDim * 4;         // bytes per row in memory
constexpr int SROWB = DW * 4;          // bytes per row of a wavefront's slice in LDS (768)
constexpr int SLICE = BN * SROWB;      // 12,288
constexpr int KPF = 4;                 // K operands in flight from LDS
// a pass restarts when a score exceeds its reference by 2^kTauLog2 (exp2 units)
constexpr float kTauLog2 = 64.0f;

struct Params {
    const float* Q;
    const float* K;
    const float* V;
    float* out;
    float* po;
    float* pm;
    float* pl;
    int B, NL, NI, S, chunk, row_blocks;
#ifdef XATTN_PHASE_CLOCK
    unsigned long long* clock;  // flash_f32_kernel's stamps, which this form fills in its place
#endif
};

typedef __attribute__((address_space(3))) char lds_char;
template <typename X>
__device__ inline X lds_read(lds_char* p) { return *(__attribute__((address_space(3))) X*)p; }
template <typename X>
__device__ inline void lds_write(lds_char* p, X v) { *(__attribute__((address_space(3))) X*)p = v; }

// Maxima of scores as single instructions (see xattn_flash_f32.hip).
__device__ inline float vmax(float a, float b) {
    float r;
    asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ inline float vmax3(float a, float b, float c) {
    float r;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

__device__ inline f4 mfma4(float a, float b, f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

template <bool PARTIAL>
__global__ __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(1, 1)))
void slice_f32_kernel(Params p) {
    // per wavefront three K slices, then the score exchange (three buffers of
    // one float4 per lane and wavefront) and the restart flag
    constexpr int XCH = NW * 3 * SLICE;
    constexpr int FLAG = XCH + 3 * NW * 1024;
    __shared__ __attribute__((aligned(16))) char lds[FLAG + 16];

    XATTN_STAMP(clk_start);
#ifdef XATTN_PHASE_CLOCK
    const unsigned long long rt_start = __builtin_amdgcn_s_memrealtime();
#endif
    const int item = xcd_remap(blockIdx.x, gridDim.x);
    const int rb = item % p.row_blocks;
    const int bs = item / p.row_blocks;
    const int split = bs % p.S;
    const int b = bs / p.S;

    const int tid = threadIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int j = lane & 15, g = lane >> 4;
    const int q0 = rb * BM;

    int k0 = 0, k1 = p.NI;
    if (PARTIAL) {
        k0 = split * p.chunk;
        k1 = min(k0 + p.chunk, p.NI);
    }
    auto out_row = [&](int q) {
        return PARTIAL ? p.po + (((size_t)b * p.NL + q) * p.S + split) * kDim
                       : p.out + ((size_t)b * p.NL + q) * kDim;
    };
    if (k0 >= k1) {
        // Empty key range: sentinel partials (kernel_splitk.cu:62-71) or, for
        // a full-range launch with N_input == 0, a zero output.
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int q = q0 + 4 * g + i;
            if (q >= p.NL) continue;
#pragma unroll
            for (int T = 0; T < NT; ++T)
                *(f4*)(out_row(q) + DW * w + 64 * T + 4 * j) = (f4){0.f, 0.f, 0.f, 0.f};
        }
        if (PARTIAL && w == 0 && g == 0 && q0 + j < p.NL) {
            const size_t pi = ((size_t)b * p.NL + q0 + j) * p.S + split;
            p.pm[pi] = -FLT_MAX;
            p.pl[pi] = 0.f;
        }
        return;
    }
    __builtin_assume(k1 - k0 >= 1);
    const int nk = k1 - k0;
    const int ntiles = (nk + BN - 1) / BN;
    __builtin_assume(ntiles >= 1);

    const char* Kb = (const char*)(p.K + (size_t)b * p.NI * kDim);
    const char* Vb = (const char*)(p.V + (size_t)b * p.NI * kDim);
    // Tile t's rows are the keys from win(t) on: k0 + 16 t, except that a
    // partial last tile is shifted back to end at k1 (its first rows repeat
    // keys of the tile before; the softmax masks them), and a range shorter
    // than a tile keeps its window at k0 with the rows past the range
    // re-reading its last row (masked too).  Every row read is a key of
    // [k0, k1).
    auto win = [&](int t) { return nk >= BN ? min(k0 + BN * t, k1 - BN) : k0; };
    auto rsrc = [&](const char* base, int t) {
        return __builtin_amdgcn_make_buffer_rsrc((void*)uniform_ptr(base + (size_t)win(t) * ROWB),
                                                 (short)0, 0x7fffffff, 0x00027000);
    };
    const int last = min(nk, BN) - 1;

    // A wavefront's K slice of 16 rows comes by DMA into its own LDS slice:
    // 16-byte pieces u = 64 m + lane, 48 per row, consecutive lanes on
    // consecutive bytes (loaded straight into the operand's layout the lanes
    // of a quad would lie on four rows and take four times as long).  Piece c
    // of row r sits at place c ^ r of its row, so that the 16 rows of an
    // operand read fall on distinct banks.
    int goff[NCH];
#pragma unroll
    for (int m = 0; m < NCH; ++m) {
        const int u = 64 * m + lane, r = u / 48, c = u % 48;
        goff[m] = ROWB * min(r, last) + 4 * DW * w + 16 * (c ^ r);
    }
    lds_char* const L = (lds_char*)lds;
    lds_char* const slice = L + w * 3 * SLICE;
    const unsigned slice0 = lds_u32(lds) + w * 3 * SLICE;
    auto ksrc = [&](int t) { return dma_base(Kb + (size_t)win(min(t, ntiles - 1)) * ROWB); };
    auto dma_k = [&](DmaSrc src, unsigned buf, int m) {
        dma16_m0<0>(src, goff[m], slice0 + buf + 1024 * m);
    };
    // operand read: lane (j, g) takes row j, piece 4 u + g
    int srd[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) srd[u] = SROWB * j + 16 * ((4 * u + g) ^ j);
    // V operand straight from memory: lane (j, g) takes V[4 g + r][64 T + 4 j ..],
    // 256 contiguous bytes per 16 lanes
    int voff[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) voff[r] = ROWB * min(4 * g + r, last) + 4 * DW * w + 16 * j;

    f4 vr[4 * NT];     // V operands of a tile: n = NT r + T
    auto load_v = [&](auto rs, int n) {
        vr[n] = __builtin_bit_cast(
            f4, __builtin_amdgcn_raw_buffer_load_b128(rs, voff[n / NT] + 256 * (n % NT), 0, 0));
    };

    lds_char* const xwr = L + XCH + w * 1024 + 16 * lane;
    lds_char* const xrd = L + XCH + 16 * lane;
    volatile __attribute__((address_space(3))) int* flag =
        (volatile __attribute__((address_space(3))) int*)(L + FLAG);
    if (tid == 0) *flag = 0;

    const float c2 = kLog2e / sqrtf((float)kDim);
    const float tau_raw = kTauLog2 / c2;
    // Softmax state per lane, as in flash_f32_kernel: weights exp2((s - m_ref) c2)
    // with m_ref fixed for a pass; a score over the bound discards the pass.
    float m_true = -FLT_MAX, m_ref = -FLT_MAX, bound = -FLT_MAX, lsum;
    bool ref_set = false;
    unsigned long long over;
    f4 acc[NT][4];
    f4 qr[NU], kf[KPF], s, sh[NW];
    float pw[4];

    auto read_k = [&](unsigned buf, int u) {
        kf[u % KPF] = lds_read<f4>(slice + buf + srd[u & 3] + 256 * (u >> 2));
    };
    auto qk_group = [&](int u) {
        const f4 k4 = kf[u % KPF];
        if (u == 0) s = (f4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < 4; ++c) s = mfma4(k4[c], qr[u][c], s);
    };
    auto pv_group = [&](int n) {
#pragma unroll
        for (int c = 0; c < 4; ++c)
            acc[n % NT][c] = mfma4(pw[n / NT], vr[n][c], acc[n % NT][c]);
    };
    auto read_shares = [&](int buf) {
#pragma unroll
        for (int d = 0; d < NW; ++d) sh[d] = lds_read<f4>(xrd + buf + d * 1024);
    };
    // Scores of tile t, the shares summed in the same order by every wavefront
    // (so all hold bit-identical scores), into the P operand (lane (j, g):
    // latent j, keys 4 g + i).  The sum and the exact maximum are kept per lane
    // and combined over a latent's four lanes at the end.
    auto softmax = [&](int t) {
        const f4 st = ((sh[0] + sh[1]) + sh[2]) + sh[3];
        const int n0 = k0 + BN * t;
        float x[4];
        if (n0 + BN <= k1) {  // a full tile (uniform branch): no key to mask
#pragma unroll
            for (int i = 0; i < 4; ++i) x[i] = st[i];
        } else {
            const int ws = win(t);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int key = ws + 4 * g + i;
                x[i] = (key >= n0 && key < k1) ? st[i] : -INFINITY;
            }
        }
        const float tmax = vmax(vmax3(x[0], x[1], x[2]), x[3]);
        if (!ref_set) {
            m_ref = wave_max16_groups(tmax);
            bound = m_ref + tau_raw;
            ref_set = true;
        }
        m_true = vmax(m_true, tmax);
        over |= __ballot(tmax > bound);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            pw[i] = fast_exp2((x[i] - m_ref) * c2);
            lsum += pw[i];
        }
    };
#define PIN() __builtin_amdgcn_sched_barrier(0)

    // The first phase is the scores; the second, all the rest of the loop
    // (output products, softmax), is the loop's time less the others': a sum
    // of its own and the stamps for it cost 90 cycles per tile more.
    XATTN_CLOCK_DECL(clk_loop = 0, pc_wait = 0, pc_qk = 0);
    for (;;) {  // passes over the key range; a second is rare
        // Q comes through the third slice (latents past NL repeat the last),
        // with K(0), K(1) and V(0) behind it.
        {
            const DmaSrc qsrc = dma_base(p.Q + ((size_t)b * p.NL + q0) * kDim);
            const int qlast = min(p.NL - q0, BM) - 1;
#pragma unroll
            for (int m = 0; m < NCH; ++m) {
                const int u = 64 * m + lane, r = u / 48, c = u % 48;
                dma16_m0<0>(qsrc, ROWB * min(r, qlast) + 4 * DW * w + 16 * (c ^ r),
                            slice0 + 2 * SLICE + 1024 * m);
            }
            const DmaSrc sk0 = ksrc(0);
#pragma unroll
            for (int m = 0; m < NCH; ++m) dma_k(sk0, 0, m);
            const DmaSrc sk1 = ksrc(1);
#pragma unroll
            for (int m = 0; m < NCH; ++m) dma_k(sk1, SLICE, m);
            const auto rv = rsrc(Vb, 0);
#pragma unroll
            for (int n = 0; n < 4 * NT; ++n) {
                load_v(rv, n);
                PIN();
            }
        }
#pragma unroll
        for (int T = 0; T < NT; ++T)
#pragma unroll
            for (int c = 0; c < 4; ++c) acc[T][c] = (f4){0.f, 0.f, 0.f, 0.f};
        lsum = 0.f;
        over = 0;
        wait_vmcnt<36>();  // Q
#pragma unroll
        for (int u = 0; u < NU; ++u)
            qr[u] = lds_read<f4>(slice + 2 * SLICE + srd[u & 3] + 256 * (u >> 2));
        __builtin_amdgcn_s_waitcnt(0xC07F);  // read before the DMA of K(2) writes there
        compiler_fence();
        XATTN_STAMP(pc_q);
#ifdef XATTN_PHASE_CLOCK
        if (clk_loop == 0) clk_loop = pc_q;
#endif
        // the first tile's scores and weights
        {
            const DmaSrc sk = ksrc(2);
            wait_vmcnt<24>();  // K(0)
#pragma unroll
            for (int u = 0; u < KPF; ++u) read_k(0, u);
#pragma unroll
            for (int u = 0; u < NU; ++u) {
                qk_group(u);
                PIN();
                if (u + KPF < NU) read_k(0, u + KPF);
                dma_k(sk, 2 * SLICE, u);
                PIN();
            }
            lds_write(xwr, s);
            XATTN_STAMP(pc_c);
            lds_barrier();
            XATTN_STAMP(pc_d);
            read_shares(0);
            wait_vmcnt<24>();  // K(1)
#pragma unroll
            for (int u = 0; u < KPF; ++u) read_k(SLICE, u);
            softmax(0);
            XATTN_CLOCK_ADD(pc_qk, pc_q, pc_c);
            XATTN_CLOCK_ADD(pc_wait, pc_c, pc_d);
        }
        // Tile t's scores, then tile t - 1's output product, under whose MFMAs
        // the scores are exchanged.  K(t + 2) and V(t) are requested.
        // The three K slices take turns (unrolled).
        auto tile = [&](int t, int turn) {  // turn = t % 3
            const unsigned kc = turn * SLICE, kn = (turn == 2 ? 0 : turn + 1) * SLICE;
            const unsigned kl = (turn == 0 ? 2 : turn - 1) * SLICE;
            const int xb = turn * (NW * 1024);
            const DmaSrc sk = ksrc(t + 2);
            XATTN_STAMP(pc_a);
#pragma unroll
            for (int u = 0; u < NU; ++u) {
                qk_group(u);
                PIN();
                if (u + KPF < NU) read_k(kc, u + KPF);
                dma_k(sk, kl, u);
                PIN();
            }
            lds_write(xwr + xb, s);
            XATTN_STAMP(pc_b);
            XATTN_CLOCK_ADD(pc_qk, pc_a, pc_b);
            const auto rv = rsrc(Vb, t);
#pragma unroll
            for (int n = 0; n < 4 * NT; ++n) {
                pv_group(n);
                PIN();
                load_v(rv, n);
                if (n == 4) {
                    XATTN_STAMP(pc_c);
                    lds_barrier();
                    XATTN_STAMP(pc_d);
                    XATTN_CLOCK_ADD(pc_wait, pc_c, pc_d);
                    read_shares(xb);
                }
                // K(t + 1): all that its reads need (the V waits in front ask
                // for more today, but only as the compiler places them)
                if (n == 8) wait_vmcnt<21>();
                if (n >= 8) read_k(kn, n - 8);
                PIN();
            }
            softmax(t);
        };
        int t = 1;
        for (; t + 2 < ntiles; t += 3) {
            tile(t, 1);
            tile(t + 1, 2);
            tile(t + 2, 0);
        }
        for (int turn = 1; t < ntiles; ++t, ++turn) tile(t, turn);
        // the last tile's output product
#pragma unroll
        for (int n = 0; n < 4 * NT; ++n) pv_group(n);
        wait_vmcnt<0>();  // the re-reads of the last tile

        // Every wavefront raises the flag (if at all) before this barrier, so
        // all of them read the same value.
        if (over != 0) *flag = 1;
        lds_barrier();
        if (!__builtin_amdgcn_readfirstlane(*flag)) break;
        // Some latent's scores outgrew its reference: clear the flag and run
        // the keys again with the reference raised to the max seen so far.
        lds_barrier();
        if (w == 0) *flag = 0;
        m_ref = wave_max16_groups(m_true);
        bound = m_ref + tau_raw;
    }

    XATTN_STAMP(clk_loop_end);
    // The latent's exact max and sum of weights over its four lanes.
    m_true = wave_max16_groups(m_true);
    lsum = wave_sum16_groups(lsum);
    // Fold the exact max back in: factor = exp(m_ref - m_true) <= 1.
    const float factor = fast_exp2((m_ref - m_true) * c2);
    float rowscale;
    if (PARTIAL) rowscale = factor;
    else rowscale = factor / (lsum * factor + 1e-6f);
    float rsc[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) rsc[i] = __shfl(rowscale, 4 * g + i);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int q = q0 + 4 * g + i;
        if (q >= p.NL) continue;
#pragma unroll
        for (int T = 0; T < NT; ++T) {
            const f4 o = (f4){acc[T][0][i], acc[T][1][i], acc[T][2][i], acc[T][3][i]} * rsc[i];
            __builtin_nontemporal_store(o, (f4*)(out_row(q) + DW * w + 64 * T + 4 * j));
        }
    }
    if (PARTIAL && w == 0 && g == 0 && q0 + j < p.NL) {
        const size_t pi = ((size_t)b * p.NL + q0 + j) * p.S + split;
        p.pm[pi] = m_true / sqrtf((float)kDim);
        p.pl[pi] = lsum * factor;
    }
#ifdef XATTN_PHASE_CLOCK
    XATTN_STAMP(clk_end);
    const unsigned long long rt_end = __builtin_amdgcn_s_memrealtime();
    if (lane == 0 && p.clock && blockIdx.x < (unsigned)kClockBlocks) {
        unsigned long long* c = p.clock + ((size_t)blockIdx.x * 8 + w) * kClockFields;
        c[0] = clk_start, c[1] = clk_loop, c[2] = clk_loop_end, c[3] = clk_end;
        c[4] = rt_start, c[5] = rt_end, c[6] = pc_wait, c[7] = pc_qk;
        c[8] = clk_loop_end - clk_loop - pc_wait - pc_qk;
    }
#endif
}

}  // namespace f32s

bool launch_slice_f32(const float* Q, const float* K, const float* V, float* out, float* po,
                      float* pm, float* pl, int B, int NL, int NI, int S, int chunk,
                      hipStream_t stream) {
    f32s::Params p;
    p.Q = Q; p.K = K; p.V = V; p.out = out; p.po = po; p.pm = pm; p.pl = pl;
    p.B = B; p.NL = NL; p.NI = NI; p.S = S; p.chunk = chunk;
    p.row_blocks = (NL + f32s::BM - 1) / f32s::BM;
#ifdef XATTN_PHASE_CLOCK
    p.clock = f32_phase_clock();
#endif
    const long long nblk = (long long)B * p.row_blocks * S;
    if (nblk <= 0) return true;
    if (nblk > 0x7fffffffLL) {
        set_error(XATTN_ERR_INVALID_VALUE, "grid of %lld workgroups too large", nblk);
        return false;
    }
    if (po)
        hipLaunchKernelGGL(f32s::slice_f32_kernel<true>, dim3((unsigned)nblk),
                           dim3(f32s::NW * kWave), 0, stream, p);
    else
        hipLaunchKernelGGL(f32s::slice_f32_kernel<false>, dim3((unsigned)nblk),
                           dim3(f32s::NW * kWave), 0, stream, p);
    return check_launch("flash_f32");
}

}  // namespace xattn

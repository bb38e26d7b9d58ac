// Streaming value projection in float32 on split operands (td_split.h): value[M, 256] = memory[M, K] . W[256, K]^T +
// bias, K = 128 or 256.
//   * One workgroup of eight wavefronts per CU (two a SIMD), each workgroup an equal share of the rows. Every
//     wavefront holds 32 output channels of W, split, in registers for the whole kernel (192 VGPRs at K = 256): W is
//     read and split once per CU, in whole rows through the LDS that the tokens take afterwards, and a step needs only
//     the tokens.
//   * A step is 32 tokens. Each wavefront brings four of them to LDS by direct loads (a KB each at K = 256), a step
//     ahead, and splits them into three bfloat16 planes there, which all eight read; the planes are double-buffered,
//     so a step costs one barrier. Of the two wavefronts of a SIMD one splits before its MFMAs and one after, so that
//     the split's VALU work (about 900 cycles a step) runs beside the other's MFMAs (6144 for the two).
//   * The product is formed transposed, D = W . tokens^T, and the rows of the output tiles are permuted, so that a
//     lane ends with 8 consecutive channels of a token (two 16-byte stores; 128 bytes by the lanes of a token).
//   * A step with a value beyond the split's range (SplitRange), or every step where W has one, runs on the float32
//     units, its operands straight from memory: 67200 x 256 x 256 161 us with an infinite weight, against 97 on the
//     register tiles (by scalar FMAs it was 8200).
//   * A plane's row is K / 8 chunks of 16 bytes, chunk c at slot c ^ (row & 15), which an LDS probe reads at the full
//     rate (525 B/ns a CU; unpermuted or padded by 16 bytes: 290).
// Bound by the MFMAs: 67200 x 256 x 256 (52.8 GFLOP in six products) 55-60 us against 100 on the float32 units, of
// which the steps 4.5 us each (1.5 PFLOP/s, the clock this load leaves; copies of the kernel without the split, the
// loads or the stores take the same) and the start, W's two round trips and its split, 8. Against the register tiles
// with v_mfma_f32_16x16x4_f32 (graph-timed us): 33600 rows 54.9 -> 32.3, 16800 32.3 -> 21.4, 8400 19.8 -> 15.4, 5000
// 13.4 -> 12.1, 177777 222 -> 117; 67201 x 128 55.9 -> 32.3, 5000 x 128 9.0 -> 8.1; below them the start costs more
// than the products save (2400 rows 8.8 -> 11.7).
#include "td_split.h"

namespace td {
namespace {

constexpr int kSplitNO = 256;
constexpr int kSplitWaves = 8;
constexpr int kSplitStep = 32;

__device__ __forceinline__ void direct_load16(const void* src, void* dst) {
    __builtin_amdgcn_global_load_lds(src, dst, 16, 0, 0);
}

// Wait until at most VM vector-memory operations of this wavefront are in flight (gfx9 encoding: vmcnt in bits 3:0 and
// 15:14, expcnt 6:4 and lgkmcnt 11:8 left alone); the empty asm statements and the scheduling barriers keep memory
// accesses on their side
template <int VM>
__device__ __forceinline__ void wait_vm() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt((VM & 15) | ((VM >> 4) << 14) | (7 << 4) | (15 << 8));
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}
// This wavefront's LDS accesses done (lgkmcnt 0, vmcnt left alone)
__device__ __forceinline__ void wait_lds() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4));
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}
// The same, then a barrier without the fence of __syncthreads (which would drain the loads in flight)
__device__ __forceinline__ void meet_lds() {
    wait_lds();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// v, which the compiler takes for a new value: what follows from it is computed where it stands instead of being kept
// in registers across the kernel's loop, which has none left
__device__ __forceinline__ int unhoisted(int v) {
    asm volatile("" : "+v"(v));
    return v;
}

// WT: W is [K, 256] as its owner stores it (C = A . W, the input gradient) instead of [256, K].
template <int KB, bool WT>
__global__ __launch_bounds__(kSplitWaves* kWave) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_split_kernel(
    GemmParams p) {
    constexpr int K = KB * 32;
    constexpr int STEP = kSplitStep;                          // two halves of 16 tokens
    constexpr int RAW_ROW = K * 4, ROWB = K * 2;              // bytes of a token row: float32, one plane
    constexpr int PLANE = STEP * ROWB, BUF = 3 * PLANE;
    constexpr int TOK = STEP / kSplitWaves;                   // tokens a wavefront loads and splits: 4
    constexpr int DL = TOK * RAW_ROW / 1024;                  // its direct loads: 4 (K = 256) or 2
    constexpr int NST = 4;                                    // its stores per step
    extern __shared__ __align__(16) unsigned char smem[];
    unsigned char* const planes = smem;                       // two buffers
    float* const bias_l = reinterpret_cast<float*>(smem + 2 * BUF + STEP * RAW_ROW);
    int* const flags = reinterpret_cast<int*>(bias_l + kSplitNO);  // [3][8]: buffer 0, buffer 1, W

    const float* __restrict__ A = static_cast<const float*>(p.a);
    const float* __restrict__ W = static_cast<const float*>(p.w);
    const float* __restrict__ bias = static_cast<const float*>(p.bias);
    float* __restrict__ C = static_cast<float*>(p.c);
    const int M = p.M;
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int r = lane & 15, kg = lane >> 4;
    const int lo = static_cast<int>(static_cast<int64_t>(blockIdx.x) * M / gridDim.x);
    const int hi = static_cast<int>(static_cast<int64_t>(blockIdx.x + 1) * M / gridDim.x);
    const int ns = (hi - lo + STEP - 1) / STEP;
    if (ns <= 0) return;  // the whole workgroup
    unsigned char* const raw = smem + 2 * BUF + wave * (TOK * RAW_ROW);

    // this wavefront's tokens of step i into its own raw rows (steps past the last re-read the last rows, unused)
    auto issue = [&](int i) {
        const int m0 = lo + STEP * (i < ns ? i : ns - 1) + wave * TOK;
#pragma unroll
        for (int j = 0; j < DL; ++j) {
            const int q = j * kWave + lane;
            int m = m0 + q / (RAW_ROW / 16);
            m = m < hi ? m : hi - 1;
            direct_load16(A + static_cast<size_t>(m) * K + (q % (RAW_ROW / 16)) * 4, raw + j * 1024);
        }
    };
    // split them into plane buffer i % 2
    auto split = [&](int i) {
        unsigned char* const dst = planes + (i & 1) * BUF;
        const int ln = unhoisted(lane);
        SplitRange range;
#pragma unroll
        for (int j = 0; j < DL; ++j) {
            const int q = j * kWave + ln;
            const f32x4 x = *reinterpret_cast<const f32x4*>(raw + q * 16);
            const int row = wave * TOK + q / (RAW_ROW / 16), c = q % (RAW_ROW / 16);
            bf16x4 h, m, l;
            split3(x, h, m, l);
            range.add(x);
            unsigned char* const at = dst + row * ROWB + ((((c >> 1) ^ (row & 15)) << 4) | ((c & 1) << 3));
            *reinterpret_cast<bf16x4*>(at) = h;
            *reinterpret_cast<bf16x4*>(at + PLANE) = m;
            *reinterpret_cast<bf16x4*>(at + 2 * PLANE) = l;
        }
        const bool any = __any(range.beyond());
        if (lane == 0) flags[(i & 1) * kSplitWaves + wave] = any;
    };

    // the channels of this wavefront, rotated by workgroup so that the CUs of an XCD start on different parts of W
    const int c0 = 32 * ((wave + static_cast<int>(blockIdx.x / kXcds)) & 7);
    const float bias_v = bias != nullptr && tid < kSplitNO ? bias[tid] : 0.f;
    // W, 16 channels of each wavefront at a time, in whole rows through the LDS that the tokens take afterwards: each
    // wavefront reads back what it brought, so no barrier
    u32x4 wf[3][2][KB];
    {
        constexpr int WDL = 16 * RAW_ROW / 1024;                       // direct loads: 16 (K = 256) or 8
        unsigned char* const wl = smem + wave * (16 * RAW_ROW);
        SplitRange range;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            // tile t's row j is channel c0 + 8 (j / 4) + 4 t + j % 4
#pragma unroll
            for (int j = 0; j < WDL; ++j) {
                const int q = j * kWave + lane;
                if constexpr (WT) {  // slot q: k row q / 4, channels of the tile's rows 4 (q % 4) on
                    direct_load16(W + static_cast<size_t>(q >> 2) * kSplitNO + c0 + 8 * (q & 3) + 4 * t, wl + j * 1024);
                } else {  // slot q: row q / (K / 4); the row's 16-byte chunk c at slot c ^ row
                    const int row = q / (K / 4), c = (q % (K / 4)) ^ row;
                    direct_load16(W + static_cast<size_t>(c0 + 8 * (row >> 2) + 4 * t + (row & 3)) * K + c * 4,
                                  wl + j * 1024);
                }
            }
            wait_vm<0>();
#pragma unroll
            for (int kb = 0; kb < KB; ++kb) {
                f32x4 x[2];
                const int k = kb * 32 + kg * 8;
                if constexpr (WT) {
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        x[e >> 2][e & 3] = *reinterpret_cast<const float*>(wl + (k + e) * 64 + r * 4);
                } else {
#pragma unroll
                    for (int e = 0; e < 2; ++e)
                        x[e] = *reinterpret_cast<const f32x4*>(wl + r * RAW_ROW + (((k / 4 + e) ^ r) << 4));
                }
                range.add(x[0]);
                range.add(x[1]);
                bf16x4 part[2][3];
#pragma unroll
                for (int e = 0; e < 2; ++e) split3(x[e], part[e][0], part[e][1], part[e][2]);
#pragma unroll
                for (int o = 0; o < 3; ++o)
                    wf[o][t][kb] = __builtin_bit_cast(
                        u32x4, __builtin_shufflevector(part[0][o], part[1][o], 0, 1, 2, 3, 4, 5, 6, 7));
            }
            wait_lds();
        }
        const bool any = __any(range.beyond());
        if (lane == 0) flags[2 * kSplitWaves + wave] = any;
    }
    if (tid < kSplitNO) bias_l[tid] = bias_v;
    __builtin_amdgcn_s_barrier();  // W's LDS is free
    issue(0);
    wait_vm<0>();
    split(0);
    wait_lds();
    issue(1);
    meet_lds();
    auto flagged = [&](int which) {
        const u32x4* f = reinterpret_cast<const u32x4*>(flags + which * kSplitWaves);
        const u32x4 v = f[0] | f[1];
        return __builtin_amdgcn_readfirstlane(static_cast<int>(v[0] | v[1] | v[2] | v[3])) != 0;
    };
    const bool w_beyond = flagged(2);

    auto product = [&](int i) {
        const int rows = min(hi - (lo + STEP * i), STEP);
        // 16 tokens' results: lane r = token, acc[t] the channels c0 + 8 kg + 4 t on
        auto put = [&](int sh, const f32x4 (&acc)[2]) {
            if (16 * sh + r < rows) {
                float* const out = C + static_cast<size_t>(lo + STEP * i + 16 * sh) * kSplitNO;  // uniform
                const int at = unhoisted(r * kSplitNO + c0 + 8 * kg);
#pragma unroll
                for (int t = 0; t < 2; ++t)
                    *reinterpret_cast<f32x4*>(out + at + 4 * t) =
                        acc[t] + *reinterpret_cast<const f32x4*>(bias_l + (at & (kSplitNO - 1)) + 4 * t);
            }
        };
        if (w_beyond || flagged(i & 1)) {  // the step on the float32 units, the operands from memory
            const int rr = unhoisted(r), kk = unhoisted(kg * 4);
            const int m = lo + STEP * i + rr, ch = c0 + 8 * (rr >> 2) + (rr & 3);  // tile t's row r: channel ch + 4 t
            const float* const a[2] = {A + static_cast<size_t>(min(m, hi - 1)) * K + kk,
                                       A + static_cast<size_t>(min(m + 16, hi - 1)) * K + kk};
            f32x4 acc[2][2], x[2], w[2];
#pragma unroll
            for (int sh = 0; sh < 2; ++sh) acc[sh][0] = acc[sh][1] = f32x4{0.f, 0.f, 0.f, 0.f};
            auto load = [&](int k) {
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    x[t] = *reinterpret_cast<const f32x4*>(a[t] + k);
                    if constexpr (WT) {
#pragma unroll
                        for (int e = 0; e < 4; ++e) w[t][e] = W[static_cast<size_t>(k + kk + e) * kSplitNO + ch + 4 * t];
                    } else {
                        w[t] = *reinterpret_cast<const f32x4*>(W + static_cast<size_t>(ch + 4 * t) * K + k + kk);
                    }
                }
            };
            load(0);
#pragma unroll 1
            for (int k = 16; k <= K; k += 16) {
                const f32x4 xc[2] = {x[0], x[1]}, wc[2] = {w[0], w[1]};
                load(min(k, K - 16));  // in flight during the MFMAs
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int sh = 0; sh < 2; ++sh)
#pragma unroll
                        for (int t = 0; t < 2; ++t)
                            acc[sh][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(wc[t][e], xc[sh][e], acc[sh][t], 0, 0, 0);
            }
            put(0, acc[0]);
            put(1, acc[1]);
            wait_vm<0>();
            return;
        }
        const unsigned char* const st = planes + (i & 1) * BUF;
        auto fragments = [&](u32x4 (&x)[3], int sh, int kb) {
#pragma unroll
            for (int o = 0; o < 3; ++o)
                x[o] = *reinterpret_cast<const u32x4*>(st + o * PLANE + (sh * 16 + r) * ROWB +
                                                       (((kb * 4 + kg) ^ r) << 4));
        };
        u32x4 x[2][3];  // a block's fragments are read while the one before it is in the MFMAs
        fragments(x[0], 0, 0);
#pragma unroll
        for (int sh = 0; sh < STEP / 16; ++sh) {
            if (sh > 0 && rows <= sh * 16) break;
            f32x4 acc[2];
#pragma unroll
            for (int t = 0; t < 2; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kb = 0; kb < KB; ++kb) {
                const u32x4 (&xc)[3] = x[kb & 1];
#pragma unroll
                for (int q = 0; q < 6; ++q) {
                    if (q == 2) {
                        __builtin_amdgcn_sched_barrier(0);
                        if (kb + 1 < KB) fragments(x[(kb + 1) & 1], sh, kb + 1);
                        else if (sh + 1 < STEP / 16) fragments(x[(kb + 1) & 1], sh + 1, 0);
                        __builtin_amdgcn_sched_barrier(0);
                    }
#pragma unroll
                    for (int t = 0; t < 2; ++t) acc[t] = KBlock<bf16>::mma(wf[kSplitA[q]][t][kb], xc[kSplitB[q]], acc[t]);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            put(sh, acc);
        }
    };
    // Step i + 1's rows were requested before step i - 1's stores (the wavefronts that split first) or step i's
    // (those that split last): NST stores may stay in flight when they are read. Only the last step has fewer stores,
    // and no split follows it.
    const bool first = wave < kSplitWaves / 2;
    auto advance = [&](int i) {
        split(i + 1);
        wait_lds();  // its raw rows are read
        issue(i + 2);
    };
    for (int i = 0; i < ns; ++i) {
        const bool more = i + 1 < ns;
        if (first && more) {
            if (i == 0) wait_vm<0>();
            else wait_vm<NST>();
            advance(i);
        }
        product(i);
        if (more) {
            if (!first) {
                wait_vm<NST>();
                advance(i);
            }
            meet_lds();
        }
    }
    wait_vm<0>();  // the last direct loads land before the workgroup gives its LDS back
}

template <int KB, bool WT>
int go_split(GemmParams p, hipStream_t stream) {
    constexpr int K = KB * 32;
    constexpr size_t lds = static_cast<size_t>(2) * 3 * kSplitStep * K * 2 + static_cast<size_t>(kSplitStep) * K * 4 +
                           kSplitNO * 4 + 3 * kSplitWaves * 4;
    static std::atomic<uint64_t> done{0};
    const hipError_t attr =
        allow_dynamic_lds(reinterpret_cast<const void*>(gemm_split_kernel<KB, WT>), static_cast<int>(lds), done);
    if (attr != hipSuccess)
        return set_error(-3, "value_proj: LDS size attribute refused: %s", hipGetErrorString(attr));
    int64_t grid = (static_cast<int64_t>(p.M) + kSplitStep - 1) / kSplitStep;
    const int cus = cu_count();
    if (grid > cus) grid = cus;
    hipLaunchKernelGGL((gemm_split_kernel<KB, WT>), dim3(static_cast<unsigned>(grid)), dim3(kSplitWaves * kWave), lds,
                       stream, p);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : set_error(-3, "value_proj launch failed: %s", hipGetErrorString(e));
}

}  // namespace

// The bias is read element by element; the output is row-major, in 16-byte stores. Eight wavefronts' registers hold W of
// 256 x 256 in its three parts and no wider one. In tiles, W through LDS as well, the split lost about as often as it won
// at other widths (128 x 128: 16800 x 384 x 384 60.5 -> 48.3 us, but x 512 102 -> 113, 8400 x 384 36.9 -> 40.2).
bool gemm_split_fits(const GemmParams& p) {
    const uintptr_t al =
        reinterpret_cast<uintptr_t>(p.a) | reinterpret_cast<uintptr_t>(p.w) | reinterpret_cast<uintptr_t>(p.c);
    return p.NO == kSplitNO && (p.K == 128 || p.K == 256) && p.M > 0 && al % 16 == 0 && p.hm_D == 0;
}

bool gemm_split_pays(const GemmParams& p) { return split_size_pays(p.M, p.K) && gemm_split_fits(p); }

int launch_gemm_split(GemmParams p, hipStream_t stream, bool w_stored) {
    if (!gemm_split_fits(p)) return set_error(-1, "value_proj: the split kernel does not take this shape");
    if (w_stored) return p.K == 256 ? go_split<8, true>(p, stream) : go_split<4, true>(p, stream);
    return p.K == 256 ? go_split<8, false>(p, stream) : go_split<4, false>(p, stream);
}

}  // namespace td

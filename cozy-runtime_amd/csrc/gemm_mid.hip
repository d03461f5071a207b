// The int8, fp8 rowwise and MXFP8 GEMMs on tiles between the narrow ones and the 256-row ones:
// one workgroup of 8 waves a CU owns a kTM x kTN tile, chosen so that the grid's rounds over the
// 256 CUs hold as little padding as the shapes allow. The epilogues are the other tiles' (int8 the
// CPU law, internal/int8_linear.py:445-448 and :276; fp8 (acc·xs)·ws + bias in float32; MX acc +
// bias), optionally then tanh-GELU.
//
// A grid of a few hundred tiles runs one round, so its time is one tile's: K/128 steps at what a
// step costs, and that is the latency of its loads unless several steps are in flight. The two
// operands come by LDS-DMA in whole 128-byte lines into a ring of kStages steps that fills the CU's
// LDS (rows x columns: 6 steps of 32x64 to 64x128, 5 of 96x128, 4 of 128x128 and 160x128, 3 of 96x256
// to 160x256, 2 of 192x256; MX, with its scales, 5 of 32x64 and 2 of 160x256; two co-resident
// workgroups of the narrow tiles hold 2 each). Waves are
// 2 (rows) x 4 (columns); the MFMA's A operand is the W tile and its B operand the X tile, so each
// lane's four results are four consecutive output columns of one row. int8 runs on
// v_mfma_i32_16x16x64_i8, fp8 and MX on v_mfma_scale_f32_16x16x128_f8f6f4, a step's K in the same
// order as the narrow tiles', so int8 and fp8 outputs are theirs bit for bit.
//
// Bound: the step. Its bytes go into the LDS and its fragments come out at ~50 KB a us and CU whatever
// the tile (compute alone 0.75 us of 128x256's 0.95 us step, DMA alone 0.5 from L2 and 0.9 with W from
// HBM), and no unit is full: at int8 1179x9216x3072 and fp8 300x14336x4096 the MFMAs are busy 45 and
// 34% of the time, fragment reads 20 and 25% without a bank conflict, and a wave waits 40% of its life.
// Measured against the narrow and 256-row tiles (us, graph replays over weights past the MALL,
// before / after): fp8 M=300 N=14336 K=4096 39.9 / 27.7, M=1024 N=9216 K=3072 68.6 / 37.7, M=1500
// N=3072 K=12288 92.1 / 66.5, M=3072 N=3072 K=3072 58.5 / 37.2; int8 M=642 N=7688 K=3840 39.4 /
// 29.6; MX, which had 256-row tiles only, M=16 N=3072 K=3072 34.6 / 11.0, M=128 42.0 / 12.0, M=400
// N=1024 K=12288 147 / 34.3, M=1024 N=3072 K=3072 44.4 / 21.8.
#include "gemm_tile.h"

namespace cozyq {
namespace {

constexpr int kMidThreads = 512;
constexpr int kMidStep = 128;              // K bytes a step
constexpr int kMidLds = 160 * 1024;
constexpr int kMidEpi = 1024 + 512 + 1024;  // weight scales, biases and row scales of a tile

template <int kKind, int kTM, int kTN>
struct Mid {
    static constexpr int kStage = (kTM + kTN) * kMidStep;
    // MX: E8M0 bytes come 16 a row (four steps') at a time, 64 rows a wave, into one of kSlots
    // blocks: the steps in flight span two (six stages: three) of them.
    static constexpr int kXGroups = (kTM + 63) / 64;
    static constexpr int kGroups = kKind == kMx ? kXGroups + kTN / 64 : 0;
    static constexpr int fit(int slots) { return (kMidLds - kMidEpi - slots * kGroups * 1024) / kStage; }
    static constexpr int slots(int stages) { return stages == 6 ? 3 : 2; }
    static constexpr int bytes(int stages) { return stages * kStage + slots(stages) * kGroups * 1024 + kMidEpi; }
    static constexpr int kMost = fit(3) >= 6 ? 6 : fit(2) > 5 ? 5 : fit(2);
    // One step less where it lets a CU hold two (MX 32x64: K=3072 N=9216 M=65 19.9 us with six, 15.7).
    static constexpr int kStages = kMost == 6 && 2 * bytes(6) > kMidLds && 2 * bytes(5) <= kMidLds ? 5 : kMost;
    static constexpr int kSlots = slots(kStages);
    static constexpr int kBytes = bytes(kStages);
    static constexpr int kHeld = kMidLds / kBytes;  // workgroups a CU's LDS holds
    static constexpr int kBlocks = (kTM + kTN) / 8;    // 8-row loads a step, over 8 waves
    static constexpr int kEach = kBlocks / 8;          // every wave's
    static constexpr int kExtra = kBlocks % 8;         // waves with one more
};

struct MidArgs {
    const uint8_t *x, *w;
    const float *xs, *ws;
    const uint8_t *xe, *we;
    const uint16_t* bias;
    uint16_t* out;
    int64_t ldo;
    int M, N, K, tiles_m, tiles_n, out_half, epilogue;
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t mid_view(const void* base, int64_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0,
                                             bytes > 0x7fffffff ? 0x7fffffff : static_cast<int>(bytes), 0x00020000);
}

template <int kKind, int kTM, int kTN, bool kOutHalf, bool kBias, int kEpi, typename Acc>
__device__ __forceinline__ void mid_store(const MidArgs& p, const uint8_t* epi, const Acc (&acc)[kTN / 64][kTM / 32],
                                          int m0, int n0, int wm, int wn, int fr, int fq) {
    const float* ws = reinterpret_cast<const float*>(epi);
    const uint8_t* bias = epi + 1024;
    const float* xs = reinterpret_cast<const float*>(epi + 1536);
    const int left = p.N - n0;
#pragma unroll
    for (int j = 0; j < kTM / 32; ++j) {
        const int ml = wm * (kTM / 2) + j * 16 + fr;
        if (m0 + ml >= p.M) continue;
        const float xsm = kKind == kMx ? 1.0f : xs[ml];
        uint16_t* row = p.out + static_cast<int64_t>(m0 + ml) * p.ldo + n0;
#pragma unroll
        for (int i = 0; i < kTN / 64; ++i) {
            const int c = wn * (kTN / 4) + i * 16 + 4 * fq;
            if (c >= left) continue;  // N % 8 == 0: c .. c + 3 are all in
            float4 w4 = make_float4(1.0f, 1.0f, 1.0f, 1.0f);
            if constexpr (kKind != kMx) w4 = *reinterpret_cast<const float4*>(ws + c);
            const float wv[4] = {w4.x, w4.y, w4.z, w4.w};
            uint2 b2 = make_uint2(0, 0);
            if constexpr (kBias) b2 = *reinterpret_cast<const uint2*>(bias + 2 * c);
            float v[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                v[r] = static_cast<float>(acc[i][j][r]);
                if constexpr (kKind != kMx) v[r] = __fmul_rn(__fmul_rn(v[r], xsm), wv[r]);
            }
            uint2 o;
            if constexpr (kKind == kInt8) {
                o = make_uint2(finish2<kOutHalf, kBias, kEpi>(v[0], v[1], b2.x), finish2<kOutHalf, kBias, kEpi>(v[2], v[3], b2.y));
            } else {
                if constexpr (kBias) {
                    v[0] = __fadd_rn(v[0], low_of<kOutHalf>(b2.x));
                    v[1] = __fadd_rn(v[1], high_of<kOutHalf>(b2.x));
                    v[2] = __fadd_rn(v[2], low_of<kOutHalf>(b2.y));
                    v[3] = __fadd_rn(v[3], high_of<kOutHalf>(b2.y));
                }
                o = make_uint2(finish2_float<kOutHalf, kEpi>(v[0], v[1]), finish2_float<kOutHalf, kEpi>(v[2], v[3]));
            }
            *reinterpret_cast<uint2*>(row + c) = o;
        }
    }
}

template <int kKind, int kTM, int kTN>
__global__ __launch_bounds__(kMidThreads, 1) void mid_kernel(const MidArgs p) {
    using T = Mid<kKind, kTM, kTN>;
    static_assert(kTM % 32 == 0 && kTN % 64 == 0 && kTM <= 256 && kTN <= 256, "tile");
    static_assert(T::kStages >= 2 && (T::kStages - 2) * (T::kEach + 1) < 64, "ring");
    static_assert(T::kGroups <= 8, "a scale group a wave");
    constexpr int kBI = kTN / 64, kBJ = kTM / 32;  // a wave's 16x16 blocks: n by m
    constexpr int kNeed = kTM * kMidStep;          // W's part of a stage
    __shared__ __attribute__((aligned(1024))) uint8_t lds[T::kBytes];
    uint8_t* const scales = lds + T::kStages * T::kStage;
    uint8_t* const epi = scales + T::kSlots * T::kGroups * 1024;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 2, wn = wave & 3;
    const int M = p.M, N = p.N, K = p.K;
    // Workgroup b runs on XCD b % 8: each XCD takes a contiguous run of tiles, M-tiles fastest, so
    // an N-tile's weight panel is read into one XCD's L2 once (1024 x 9216 x 3072 in 252 tiles with
    // the panels spread over the XCDs fetched 218 MB instead of 31).
    const int b = blockIdx.x, each = gridDim.x >> 3, more = gridDim.x & 7, x = b & 7;
    const int t = x * each + min(x, more) + (b >> 3);
    const int tm = t % p.tiles_m, tn = t / p.tiles_m;
    const int m0 = __builtin_amdgcn_readfirstlane(tm * kTM), n0 = __builtin_amdgcn_readfirstlane(tn * kTN);
    const __amdgpu_buffer_rsrc_t xr = mid_view(p.x + static_cast<int64_t>(m0) * K, static_cast<int64_t>(M - m0) * K);
    const __amdgpu_buffer_rsrc_t wr = mid_view(p.w + static_cast<int64_t>(n0) * K, static_cast<int64_t>(N - n0) * K);
    const int kb = K / 32;  // MX: E8M0 bytes a row
    __amdgpu_buffer_rsrc_t er = xr;
    int eoff = 0;
    if constexpr (kKind == kMx) {
        const bool xside = wave < T::kXGroups;
        const int row = 64 * (xside ? wave : wave - T::kXGroups) + lane;
        er = xside ? mid_view(p.xe + static_cast<int64_t>(m0) * kb, static_cast<int64_t>(M - m0) * kb)
                   : mid_view(p.we + static_cast<int64_t>(n0) * kb, static_cast<int64_t>(N - n0) * kb);
        eoff = row * kb;  // past the operand's rows: out of range, zeros
    }
    const int nk = (K + kMidStep - 1) / kMidStep;

    // Load j of a wave brings row block 8j + wave of the stage's [X rows | W rows]: 8 rows of 128
    // bytes, lane l at row l/8 and physical chunk l%8 (logical chunk swz).
    constexpr int kMost = T::kEach + (T::kExtra > 0 ? 1 : 0);
    int off[kMost], chunk[kMost];
#pragma unroll
    for (int j = 0; j < kMost; ++j) {
        const int row = (8 * j + wave) * 8 + (lane >> 3);  // of the stage
        chunk[j] = 16 * swz(row, lane & 7);
        off[j] = (row < kTM ? row : row - kTM) * K + chunk[j];
    }
    auto issue = [&](int ks) {
        uint8_t* base = lds + (ks % T::kStages) * T::kStage;
        const int k0 = ks * kMidStep;
        // Ahead of the first of their four steps, so whoever waits for that step waits for them;
        // the waits count a step's other loads, and so ask a little more while these are newer.
        if constexpr (kKind == kMx) {
            if (ks % 4 == 0 && wave < T::kGroups) {
                const uint32_t at = 4 * ks < kb ? static_cast<uint32_t>(eoff + 4 * ks) : kOutOfRange;
                uint8_t* const dst = scales + ((ks / 4) % T::kSlots * T::kGroups + wave) * 1024;
                __builtin_amdgcn_raw_ptr_buffer_load_lds(er, (LdsPtr*)dst, 16, at, 0, 0, 0);
            }
        }
#pragma unroll
        for (int j = 0; j < kMost; ++j) {
            if (j == T::kEach && wave >= T::kExtra) break;  // uniform
            const uint32_t at = k0 + chunk[j] < K ? static_cast<uint32_t>(off[j] + k0) : kOutOfRange;
            // A load's rows are all X or all W: known for most j, else by the wave.
            constexpr int kXBlocks = kTM / 8;
            uint8_t* const dst = base + (8 * j + wave) * 1024;
            if (8 * j + 7 < kXBlocks || (8 * j < kXBlocks && 8 * j + wave < kXBlocks))
                __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (LdsPtr*)dst, 16, at, 0, 0, 0);
            else
                __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (LdsPtr*)dst, 16, at, 0, 0, 0);
        }
    };

    // The epilogue's operands first (LDS-DMA of 4 bytes a lane).
    if (wave < 4) {
        const int c = 64 * wave + lane;
        if constexpr (kKind != kMx) {
            __builtin_amdgcn_raw_ptr_buffer_load_lds(mid_view(p.ws + n0, 4 * static_cast<int64_t>(N - n0)), (LdsPtr*)(epi + 256 * wave), 4, 4 * c, 0, 0, 0);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(mid_view(p.xs + m0, 4 * static_cast<int64_t>(M - m0)), (LdsPtr*)(epi + 1536 + 256 * wave), 4, 4 * c, 0, 0, 0);
        }
        if (p.bias != nullptr && wave < 2)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(mid_view(p.bias + n0, 2 * static_cast<int64_t>(N - n0)), (LdsPtr*)(epi + 1024 + 256 * wave), 4, 4 * c, 0, 0, 0);
    }
#pragma unroll
    for (int ks = 0; ks < T::kStages - 1; ++ks) issue(ks);

    typedef std::conditional_t<kKind == kInt8, i32x4, f32x4> Acc;
    Acc acc[kBI][kBJ];
#pragma unroll
    for (int i = 0; i < kBI; ++i)
#pragma unroll
        for (int j = 0; j < kBJ; ++j) acc[i][j] = Acc{0, 0, 0, 0};

    const int fr = lane & 15, fq = lane >> 4;
    auto stage = [&](int ks) { return lds + (ks % T::kStages) * T::kStage; };
    auto x_piece = [&](int ks, int j, int c) {
        const int r = wm * (kTM / 2) + j * 16 + fr;
        return *reinterpret_cast<const i32x4*>(stage(ks) + r * kMidStep + swz(r, c) * 16);
    };
    auto w_piece = [&](int ks, int i, int c) {
        const int r = wn * (kTN / 4) + i * 16 + fr;
        return *reinterpret_cast<const i32x4*>(stage(ks) + kNeed + r * kMidStep + swz(r, c) * 16);
    };
    // Step ks landed (this wave's share; the barrier makes every wave's visible). Steps past the last
    // are issued too (zeros into slots nothing reads), so the counts hold at every wait.
    auto landed = [&]() {
        fence();
        if (wave < T::kExtra) wait_vmcnt<(T::kStages - 2) * (T::kEach + 1)>();
        else wait_vmcnt<(T::kStages - 2) * T::kEach>();
        wait_lgkmcnt0();
        __builtin_amdgcn_s_barrier();
        fence();
    };
    // A step runs in two pieces. The second piece's fragments are read while the first's MFMAs run;
    // then the workgroup meets (step ks + 1 landed, every wave's reads of step ks are in registers,
    // whose slot takes step ks + kStages), and the next step's first fragments are read while the
    // second piece's MFMAs run. (Reading a whole step, then multiplying it, left the LDS and the
    // matrix cores taking turns: 128x256 0.95 us a step.)
    landed();
    issue(T::kStages - 1);
    if constexpr (kKind == kInt8) {  // pieces: the step's two K halves
        struct Half { i32x4 a[kBI], x[kBJ]; };
        auto fetch = [&](int ks, int h, Half& f) {
#pragma unroll
            for (int i = 0; i < kBI; ++i) f.a[i] = w_piece(ks, i, 4 * h + fq);
#pragma unroll
            for (int j = 0; j < kBJ; ++j) f.x[j] = x_piece(ks, j, 4 * h + fq);
        };
        auto multiply = [&](const Half& f) {
#pragma unroll
            for (int i = 0; i < kBI; ++i)
#pragma unroll
                for (int j = 0; j < kBJ; ++j) acc[i][j] = mfma_i8(f.a[i], f.x[j], acc[i][j]);
        };
        Half f0, f1;
        fetch(0, 0, f0);
        for (int ks = 0; ks < nk; ++ks) {
            fetch(ks, 1, f1);
            multiply(f0);
            landed();
            issue(ks + T::kStages);
            fetch(ks + 1, 0, f0);  // past the last step: zeros, unused
            multiply(f1);
        }
    } else {  // pieces: the X blocks' first and second half, on the same W fragments
        constexpr int kFirst = (kBJ + 1) / 2, kSecond = kBJ - kFirst;
        struct Weights { i32x8 a[kBI]; int s[kBI]; };
        struct Rows { i32x8 x[kFirst]; int s[kFirst]; };
        auto scale_at = [&](int ks, int group, int r) {  // row r of the groups from `group` on
            const uint8_t* e = scales + ((ks / 4) % T::kSlots * T::kGroups + group) * 1024;
            return static_cast<int>(*reinterpret_cast<const uint32_t*>(e + 16 * r + 4 * (ks % 4)) >> (8 * fq));
        };
        auto weights = [&](int ks, Weights& f) {
#pragma unroll
            for (int i = 0; i < kBI; ++i) {
                f.a[i] = __builtin_shufflevector(w_piece(ks, i, fq), w_piece(ks, i, fq + 4), 0, 1, 2, 3, 4, 5, 6, 7);
                if constexpr (kKind == kMx) f.s[i] = scale_at(ks, T::kXGroups, wn * (kTN / 4) + i * 16 + fr);
            }
        };
        auto rows = [&](int ks, int j0, int count, Rows& f) {
#pragma unroll
            for (int j = 0; j < kFirst; ++j) {
                if (j >= count) break;
                f.x[j] = __builtin_shufflevector(x_piece(ks, j0 + j, fq), x_piece(ks, j0 + j, fq + 4), 0, 1, 2, 3, 4, 5, 6, 7);
                if constexpr (kKind == kMx) f.s[j] = scale_at(ks, 0, wm * (kTM / 2) + (j0 + j) * 16 + fr);
            }
        };
        auto multiply = [&](const Weights& w, const Rows& f, int j0, int count) {
#pragma unroll
            for (int j = 0; j < kFirst; ++j) {
                if (j >= count) break;
#pragma unroll
                for (int i = 0; i < kBI; ++i) {
                    if constexpr (kKind == kMx) acc[i][j0 + j] = mfma_f8_scaled(w.a[i], f.x[j], acc[i][j0 + j], w.s[i], f.s[j]);
                    else acc[i][j0 + j] = mfma_f8(w.a[i], f.x[j], acc[i][j0 + j]);
                }
            }
        };
        Weights w0, w1;
        Rows r0, r1;
        weights(0, w0);
        rows(0, 0, kFirst, r0);
        auto step = [&](int ks, const Weights& w, Weights& next) {
            rows(ks, kFirst, kSecond, r1);
            multiply(w, r0, 0, kFirst);
            landed();
            issue(ks + T::kStages);
            weights(ks + 1, next);
            rows(ks + 1, 0, kFirst, r0);
            multiply(w, r1, kFirst, kSecond);
        };
        for (int ks = 0; ks < nk; ks += 2) {
            step(ks, w0, w1);
            if (ks + 1 < nk) step(ks + 1, w1, w0);
        }
    }
    wait_vmcnt<0>();  // the zero-filling loads past the last step land before the wave ends

    // The epilogue's variants, chosen by uniform branches.
#define COZYQ_STORE(H, B, E)                                                             \
    if ((p.out_half != 0) == H && (p.bias != nullptr) == B && p.epilogue == E) {            \
        mid_store<kKind, kTM, kTN, H, B, E>(p, epi, acc, m0, n0, wm, wn, fr, fq);            \
        return;                                                                          \
    }
    COZYQ_STORE(false, false, 0)
    COZYQ_STORE(false, true, 0)
    COZYQ_STORE(true, false, 0)
    COZYQ_STORE(true, true, 0)
    if constexpr (kKind != kMx) {
        COZYQ_STORE(false, false, 1)
        COZYQ_STORE(false, true, 1)
        COZYQ_STORE(true, false, 1)
        COZYQ_STORE(true, true, 1)
    }
#undef COZYQ_STORE
}

template <int kKind, int kTM, int kTN>
hipError_t launch_mid(MidArgs p, hipStream_t s) {
    p.tiles_m = (p.M + kTM - 1) / kTM;
    p.tiles_n = (p.N + kTN - 1) / kTN;
    mid_kernel<kKind, kTM, kTN><<<p.tiles_m * p.tiles_n, kMidThreads, 0, s>>>(p);
    return hipGetLastError();
}

struct MidTile {
    int rows, cols;
    int held;    // workgroups of it a CU holds
    float step;  // us a 128-byte K step
};
template <int kTM, int kTN>
constexpr MidTile mid_tile(float step) {
    static_assert(Mid<kInt8, kTM, kTN>::kHeld == Mid<kFp8, kTM, kTN>::kHeld && Mid<kInt8, kTM, kTN>::kHeld == Mid<kMx, kTM, kTN>::kHeld, "one table for every kind");
    return {kTM, kTN, Mid<kInt8, kTM, kTN>::kHeld, step};
}
constexpr MidTile kMidTiles[] = {mid_tile<32, 64>(0.24f),  mid_tile<64, 64>(0.23f),   mid_tile<64, 128>(0.43f),
                                 mid_tile<96, 128>(0.50f), mid_tile<128, 128>(0.58f), mid_tile<160, 128>(0.68f),
                                 mid_tile<96, 256>(0.83f), mid_tile<128, 256>(0.95f), mid_tile<160, 256>(1.15f),
                                 mid_tile<192, 256>(1.40f)};

template <int kKind>
hipError_t mid_by_tile(int tile, const MidArgs& p, hipStream_t s) {
    switch (tile) {
        case 0: return launch_mid<kKind, 32, 64>(p, s);
        case 1: return launch_mid<kKind, 64, 64>(p, s);
        case 2: return launch_mid<kKind, 64, 128>(p, s);
        case 3: return launch_mid<kKind, 96, 128>(p, s);
        case 4: return launch_mid<kKind, 128, 128>(p, s);
        case 5: return launch_mid<kKind, 160, 128>(p, s);
        case 6: return launch_mid<kKind, 96, 256>(p, s);
        case 7: return launch_mid<kKind, 128, 256>(p, s);
        case 8: return launch_mid<kKind, 160, 256>(p, s);
        case 9: return launch_mid<kKind, 192, 256>(p, s);
        default: return hipErrorNotSupported;
    }
}

}  // namespace

// The tile for a shape, by a model of the round fitted on MI355X (fp8 and int8, 40 shapes of M 33 to
// 2048, N 1000 to 14336, K 1280 to 12288; within ~12% of the best tile measured at each; against the
// narrow and 256-row tiles at 7434 points of M 1 to 3072, N 640 to 128256, K 1024 to 12288 its choices
// take 0.88 of their time on average and 1.09 at worst): a grid costs its rounds over the CUs, a round
// kFixed and K/128 steps of what the tile's step costs, which is its LDS traffic (the step's bytes
// written by DMA and read 1 to 3 times as fragments).
int mid_choice(int kind, int M, int N, int K) {
    constexpr int64_t kCUs = 256;
    constexpr float kFixed = 5.0f;  // us: launch, first loads, epilogue
    // The 256-row tiles (4-wave 256x192 for every kind and MX's 256x256, else 8-wave 256x256).
    constexpr float kBig256 = 1.72f, kBig192 = 1.53f;
    const int steps = (K + kMidStep - 1) / kMidStep;
    auto rounds = [&](int rows, int cols, int64_t slots) {
        const int64_t t = static_cast<int64_t>((M + rows - 1) / rows) * ((N + cols - 1) / cols);
        return static_cast<float>((t + slots - 1) / slots);
    };
    int best = -1;
    float least = 0.0f;
    constexpr int kTiles = sizeof(kMidTiles) / sizeof(kMidTiles[0]);
    for (int t = 0; t < kTiles; ++t) {
        const MidTile& m = kMidTiles[t];
        const float cost = rounds(m.rows, m.cols, kCUs * m.held) * (steps * m.step + kFixed);
        if (best < 0 || cost < least) best = t, least = cost;
    }
    const float tail = tail_columns(M, N) > 0 ? 0.45f : 0.0f;  // its last round runs as half-width tiles
    const float big = fminf((rounds(256, 256, kCUs) - tail) * (steps * kBig256 + kFixed),
                            rounds(256, 192, kCUs) * (steps * kBig192 + kFixed));
    if (0.97f * big <= least) return -1;
    // The smallest tiles' work is the narrow tiles' at short K, and where their 32x64 grid is one
    // round (K=3072 N=3072 M=77 8.5 us there and 9.0 here; K=12288 N=3072 M=48 23.7 and 29.7; but
    // M=200 39.9 and 28.3). MX has no narrow tiles.
    if (kind != kMx && kMidTiles[best].cols == 64 && (steps <= 32 || rounds(32, 64, kCUs) <= 1.0f)) return -1;
    if (kind == kMx) return best;
    const int config = gemm_config(kind == kFp8, M, N, K);
    if (config == 0 || config == 5) {
        // At short K and in several rounds what a round costs besides its steps decides: 2.6 us and a
        // tile's epilogue here, 7 there (fp8 N=12288 M=3072 K=1024 52 us on 256x192, 62 on 192x256).
        const MidTile& m = kMidTiles[best];
        const float times = rounds(m.rows, m.cols, kCUs * m.held);
        const float mid = times * (steps * m.step * m.held + 2.6f + 1.85e-4f * m.rows * m.cols);
        const float whole = config == 0 ? (rounds(256, 256, kCUs) - tail) * (steps * 1.58f + 7.0f) + 3.0f
                                        : rounds(256, 192, kCUs) * (steps * 1.38f + 6.5f) + 3.5f;
        if ((times > 1.0f || steps <= 8) && mid > 0.98f * whole) return -1;
    } else if (config >= 3 && N <= 3072 && (N + 63) / 64 % 8 == 0) {
        // A grid of hardly more narrow tiles than CUs, many M-tiles to each XCD's few weight panels,
        // runs at one tile's pace, 0.3 us a step of 64x64 and 0.22 of 32x64 (K=8192, us, mid / narrow:
        // M=384 N=3072 30.1 / 25.7, M=768 N=1536 27.5 / 23.1, M=192 N=3072 26.3 / 23.9; past the line
        // M=416 N=3072 31.5 / 36.2, M=768 N=2048 31.5 / 35.8).
        const float narrow = rounds(config == 3 ? 64 : 32, 64, 1);
        if (narrow >= 256.0f && narrow <= (N <= 1536 ? 336.0f : 320.0f)) return -1;
    }
    return best;
}

int mid_tile_size(int tile, int* rows, int* cols) {
    if (tile < 0) return -1;
    *rows = kMidTiles[tile].rows;
    *cols = kMidTiles[tile].cols;
    return tile;
}

hipError_t gemm_mid(int kind, int tile, const void* q, const float* xs, const uint8_t* qe, const void* w,
                    const float* ws, const uint8_t* we, const void* bias, void* out, int64_t ldo,
                    bool out_half, int M, int N, int K, int epilogue, hipStream_t s) {
    const MidArgs p{static_cast<const uint8_t*>(q), static_cast<const uint8_t*>(w), xs, ws, qe, we,
                    static_cast<const uint16_t*>(bias), static_cast<uint16_t*>(out), ldo, M, N, K, 0, 0,
                    out_half, epilogue};
    if (kind == kInt8) return mid_by_tile<kInt8>(tile, p, s);
    if (kind == kFp8) return mid_by_tile<kFp8>(tile, p, s);
    return mid_by_tile<kMx>(tile, p, s);
}

}  // namespace cozyq

// gdn_inproj.hip -- the GDN layer's input projection on gfx950 bf16 MFMA (ix_gdn_in_proj).
//
// For B token rows of hidden states h [B][K] and the projection weight W [N][K] (one row per
// output, as the reference's GEMV weights, src/ix_bf16_gemv.cu:36), computes
//   y = h W^T,  N = C + h_v*d_v + 2*h_v  (C = 2 h_k d_k + h_v d_v)
// with fp32 accumulation, and writes the four pieces a GDN layer consumes as bf16 (round to
// nearest even): the mixed conv input x [B][C] (columns 0..C), the output-gate logits
// z [B][h_v][d_v], and the gate and beta logits a, b [B][h_v]. This is the step to the left
// of the recurrence that the reference runs as per-token bf16 GEMVs.
//
// Prompts (many rows) run on larger tiles, in_proj_tile_kernel below; this is the decode batches'
// kernel. At decode batch sizes the product is a skinny GEMM that streams W once from HBM (about 2
// FLOP per weight byte at B = 64), so the work is moving bytes, not MFMA throughput. One
// workgroup owns a 64 x 64 output tile over the whole of K. Two producer waves copy 64-k
// stages of the tile's 64 activation rows (one wave) and 64 weight rows (the other) into a
// ring of LDS stages with direct global-to-LDS loads: every load instruction moves 1 KiB =
// 8 whole 128-byte row segments, and the loads of three stages are in flight at once.
// Eight consumer waves each own a 32 x 16 eighth of the tile and run
// v_mfma_f32_16x16x32_bf16 on operands read from the ring; they issue no LDS DMA, so the
// compiler never makes their LDS reads wait for the copies in flight. Producers and
// consumers meet at one barrier per stage. In LDS the 16-byte chunk c of tile row r sits
// at position c ^ (r & 7) of the row's 128 bytes, so the eight rows an operand read touches
// at once fall in different banks; the producers apply the swizzle by choosing which chunk
// each lane fetches. The summation order over K is fixed, so results do not depend on
// timing.
#include "gdn_common.h"

#include <algorithm>

namespace ixg {
namespace {

constexpr int kNt = 64;                 // output columns per workgroup (4 MFMA n-tiles)
constexpr int kMt = 64;                 // rows per workgroup (4 MFMA m-tiles)
constexpr int kKd = 64;                 // k per stage (two MFMA k-steps)
constexpr int kRowB = 2 * kKd;          // bytes of one tile row per stage
constexpr int kRowsPerCopy = 1024 / kRowB;          // tile rows per 1 KiB load instruction
constexpr int kHalf = 64 * kRowB;       // bytes of one operand tile per stage
constexpr int kStage = 2 * kHalf;       // activation tile, then weight tile
constexpr int kRing = 4;                // stages in the LDS ring (64 KiB)
constexpr int kCons = 8, kProd = 2;     // consumer and producer waves
constexpr int kTM = 2, kTN = 1;         // 16 x 16 output tiles per consumer wave (rows, columns)
static_assert(2 * 16 * kTM == kMt && (kCons / 2) * 16 * kTN == kNt, "the consumer waves cover the tile");
constexpr int kCopies = 2 * (64 / kRowsPerCopy) / kProd;   // load instructions per producer and stage

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) uint8_t lds_u8;

struct InProj {
    const uint16_t* h;          // [B][K]
    const uint16_t* w;          // [N][K]
    uint16_t* x;                // [B][C]
    uint16_t* z;                // [B][Z]
    uint16_t* a;                // [B][h_v]
    uint16_t* b;                // [B][h_v]
    float* y;                   // [B][N] fp32, or null
    int B, K, N, C, Z, hv;
    int n0;                     // first column of this launch
};

__device__ __forceinline__ void store_out(const InProj& p, int row, int col, float v) {
    const uint16_t u = f32_to_bf16(v);
    if (col < p.C) p.x[(size_t)row * p.C + col] = u;
    else if (col < p.C + p.Z) p.z[(size_t)row * p.Z + (col - p.C)] = u;
    else if (col < p.C + p.Z + p.hv) p.a[(size_t)row * p.hv + (col - p.C - p.Z)] = u;
    else p.b[(size_t)row * p.hv + (col - p.C - p.Z - p.hv)] = u;
    if (p.y) p.y[(size_t)row * p.N + col] = v;
}

// s_waitcnt that waits until at most N vector memory operations are outstanding, in the
// gfx9-family field layout (gfx950 here: vmcnt in bits 3:0 and 15:14, expcnt and lgkmcnt
// left at their maximum); another target would need its own encoding.
#if defined(__HIP_DEVICE_COMPILE__) && !defined(__gfx950__)
#error "wait_vmcnt encodes gfx950 s_waitcnt fields"
#endif
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

// Byte offset in an operand tile of 16-byte chunk c of row r.
__device__ __forceinline__ int ring_off(int r, int c) { return r * kRowB + ((c ^ (r & 7)) << 4); }

__global__ void __launch_bounds__((kCons + kProd) * kWave) in_proj_kernel(const InProj p) {
    __shared__ __align__(16) uint8_t lds[kRing * kStage];

    const int lane = threadIdx.x & (kWave - 1);
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int n0 = p.n0 + blockIdx.x * kNt, m0 = blockIdx.y * kMt;
    const int nst = p.K / kKd;

    if (w >= kCons) {
        // Producer: the first half of the producer waves copy activation rows, the second
        // half weight rows, kCopies load instructions each. Instruction g of a tile covers
        // rows kRowsPerCopy g .. +kRowsPerCopy-1; lane l writes position l % (kRowB / 16) of
        // row kRowsPerCopy g + l / (kRowB / 16), so it fetches chunk position ^ (row & 7) of
        // that row. Rows past the end are clamped (their results are never stored).
        const int pw = w - kCons;
        const bool act = pw < kProd / 2;
        const int g0 = (pw % (kProd / 2)) * kCopies;          // first load instruction of this wave
        const int rr = lane / (kRowB / 16), pos = lane % (kRowB / 16);
        const uint8_t* src[kCopies];
#pragma unroll
        for (int j = 0; j < kCopies; ++j) {
            const int r = kRowsPerCopy * (g0 + j) + rr;
            const int chunk = pos ^ (r & 7);
            const int row = act ? min(m0 + r, p.B - 1) : min(n0 + r, p.N - 1);
            src[j] = reinterpret_cast<const uint8_t*>(act ? p.h : p.w) + (size_t)row * p.K * 2 + chunk * 16;
        }
        lds_u8* dst = (lds_u8*)lds + (act ? 0 : kHalf) + g0 * 1024;
        // Virtual stage v goes to ring slot v % kRing; stages past the end repeat the last one,
        // so every trip issues the same number of loads.
        auto issue = [&](int v) {
            const int sv = min(v, nst - 1);
            lds_u8* d = dst + (v % kRing) * kStage;
#pragma unroll
            for (int j = 0; j < kCopies; ++j) __builtin_amdgcn_global_load_lds(src[j] + sv * kRowB, d + j * 1024, 16, 0, 0);
        };
#pragma unroll
        for (int v = 0; v < kRing - 1; ++v) issue(v);
        wait_vmcnt<kCopies * (kRing - 2)>();                   // stage 0 landed
        __builtin_amdgcn_s_barrier();
        for (int st = 0; st < nst; ++st) {
            // The slot of stage st + kRing - 1 held stage st - 1, read before this barrier.
            issue(st + kRing - 1);
            wait_vmcnt<kCopies * (kRing - 2)>();               // stage st + 1 landed
            __builtin_amdgcn_s_barrier();
        }
        __builtin_amdgcn_s_waitcnt(0);
        return;
    }

    // Consumer wave w: rows 32 (w & 1) .. +31, columns 16 (w >> 1) .. +15 of the tile.
    const int li = lane & 15, lg = lane >> 4;
    const int rbase = 16 * kTM * (w & 1), cbase = 16 * kTN * (w >> 1);
    f32x4 acc[kTM][kTN];
#pragma unroll
    for (int mt = 0; mt < kTM; ++mt)
#pragma unroll
        for (int nt = 0; nt < kTN; ++nt) acc[mt][nt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    // Operand offsets inside a stage: lane (li, lg) of k-step ks holds k = 32 ks + 8 lg .. +7
    // of its row (chunk 4 ks + lg).
    constexpr int kSteps = kKd / 32;
    int ao[kTM][kSteps], bo[kTN][kSteps];
#pragma unroll
    for (int ks = 0; ks < kSteps; ++ks) {
#pragma unroll
        for (int t = 0; t < kTM; ++t) ao[t][ks] = ring_off(rbase + 16 * t + li, 4 * ks + lg);
#pragma unroll
        for (int t = 0; t < kTN; ++t) bo[t][ks] = kHalf + ring_off(cbase + 16 * t + li, 4 * ks + lg);
    }
    lds_barrier();
    for (int st = 0; st < nst; ++st) {
        const uint8_t* sp = lds + (st % kRing) * kStage;
        bf16x8 av[kTM][kSteps], bv[kTN][kSteps];
#pragma unroll
        for (int ks = 0; ks < kSteps; ++ks) {
#pragma unroll
            for (int t = 0; t < kTM; ++t) av[t][ks] = *reinterpret_cast<const bf16x8*>(sp + ao[t][ks]);
#pragma unroll
            for (int t = 0; t < kTN; ++t) bv[t][ks] = *reinterpret_cast<const bf16x8*>(sp + bo[t][ks]);
        }
#pragma unroll
        for (int ks = 0; ks < kSteps; ++ks)
#pragma unroll
            for (int mt = 0; mt < kTM; ++mt)
#pragma unroll
                for (int nt = 0; nt < kTN; ++nt)
                    acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[mt][ks], bv[nt][ks], acc[mt][nt], 0, 0, 0);
        lds_barrier();                                          // this slot may be refilled
    }

    // acc[mt][nt][r] is output (row rbase + 16 mt + 4 lg + r, column cbase + 16 nt + li).
#pragma unroll
    for (int mt = 0; mt < kTM; ++mt)
#pragma unroll
        for (int nt = 0; nt < kTN; ++nt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = m0 + rbase + 16 * mt + 4 * lg + r, col = n0 + cbase + 16 * nt + li;
                if (row < p.B && col < p.N) store_out(p, row, col, acc[mt][nt][r]);
            }
}

// ---------------------------------------------------------------------------------------
// Many rows (prompts): the product is bound by the matrix cores, and 64 x 64 tiles re-read each
// operand so often that they ran at 402 TFLOP/s (4096 rows, hidden 2048, N = 12,352: 516 us). Here a
// workgroup owns a BM x BN tile, its waves 2 x BN / 64 of them in accumulators (256 x 256 on 8 waves
// of 128 x 64, or 128 x 128 on 4 of 64 x 64, two workgroups per CU), so that an operand row read from
// LDS serves 64 or 128 columns. Stages of 64 k go through registers into one of two LDS buffers:
// the loads of stage s + 2 and the LDS writes of stage s + 1 are issued ahead of stage s's products.
// The tile columns are whole tiles of x and z (their width is a multiple of 128); in_proj_kernel
// takes the rest. Outputs leave through LDS as whole row segments, 16 bytes a lane. Tiles are
// numbered so that an XCD (workgroup index mod 8) works on a compact block: 8 row tiles, column by
// column.
// ---------------------------------------------------------------------------------------
template <int BM, int BN>
struct Tile {
    static constexpr int kWavesM = 2, kWavesN = BN / 64, kWaves = kWavesM * kWavesN;
    static constexpr int kThreads = kWaves * kWave;
    static constexpr int kMT = BM / kWavesM / 16, kNT = 4;             // 16 x 16 tiles per wave
    static constexpr int kBuf = (BM + BN) * kRowB;                     // one stage
    static constexpr int kChunks = (BM + BN) * 8 / kThreads;           // 16-byte chunks per thread and stage
    static constexpr int kOutRow = BN * 2 + 16;                        // bytes of an output row in LDS
    static constexpr int kLds = 2 * kBuf > BM / 2 * kOutRow ? 2 * kBuf : BM / 2 * kOutRow;
};

template <int BM, int BN>
__global__ void __launch_bounds__((Tile<BM, BN>::kThreads)) __attribute__((amdgpu_waves_per_eu(2)))
in_proj_tile_kernel(const InProj p, int mt, int nt) {
    using T = Tile<BM, BN>;
    __shared__ __align__(16) uint8_t lds[T::kLds];
    const int total = mt * nt, share = (total + 7) / 8;
    const int id = (int)(blockIdx.x & 7) * share + (int)(blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= share || id >= total) return;
    const int grp = id / (8 * nt), gm = min(8, mt - 8 * grp), in = id - grp * 8 * nt;
    const int m0 = (8 * grp + in % gm) * BM, n0 = in / gm * BN;

    const int tid = threadIdx.x, lane = tid & (kWave - 1), li = lane & 15, lg = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int wm = (w & 1) * (BM / 2), wn = (w >> 1) * 64;
    const int nst = p.K / kKd;

    // Chunk c of rows r0, r0 + T / 8, ...: activation rows, then weight rows (rows past the batch
    // repeat its last one; their results are never stored).
    const int c = tid & 7, r0 = tid >> 3;
    const uint8_t* src[T::kChunks];
#pragma unroll
    for (int i = 0; i < T::kChunks; ++i) {
        const int r = r0 + i * (T::kThreads / 8);
        const bool act = i * (T::kThreads / 8) < BM;
        const int row = act ? min(m0 + r, p.B - 1) : n0 + r - BM;
        src[i] = reinterpret_cast<const uint8_t*>(act ? p.h : p.w) + (size_t)row * p.K * 2 + c * 16;
    }
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    u32x4 st[T::kChunks];
    auto load = [&](int s) {
#pragma unroll
        for (int i = 0; i < T::kChunks; ++i) st[i] = *reinterpret_cast<const u32x4*>(src[i] + (size_t)s * kRowB);
    };
    const int wo = ring_off(r0, c);                              // r0 + multiples of 8: the same swizzle
    auto put = [&](int s) {
        uint8_t* b = lds + (s & 1) * T::kBuf + wo;
#pragma unroll
        for (int i = 0; i < T::kChunks; ++i) *reinterpret_cast<u32x4*>(b + i * (T::kThreads / 8) * kRowB) = st[i];
    };

    f32x4 acc[T::kMT][T::kNT];
#pragma unroll
    for (int i = 0; i < T::kMT; ++i)
#pragma unroll
        for (int j = 0; j < T::kNT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    int ao[2], bo[2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
        ao[ks] = ring_off(wm + li, 4 * ks + lg);
        bo[ks] = BM * kRowB + ring_off(wn + li, 4 * ks + lg);
    }

    load(0);
    put(0);
    if (nst > 1) load(1);
    for (int s = 0; s < nst; ++s) {
        lds_barrier();                                           // stage s written; stage s - 1 read
        if (s + 1 < nst) put(s + 1);
        if (s + 2 < nst) load(s + 2);
        const uint8_t* b = lds + (s & 1) * T::kBuf;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            bf16x8 av[T::kMT], bv[T::kNT];
#pragma unroll
            for (int j = 0; j < T::kNT; ++j) bv[j] = *reinterpret_cast<const bf16x8*>(b + bo[ks] + j * 16 * kRowB);
#pragma unroll
            for (int i = 0; i < T::kMT; ++i) av[i] = *reinterpret_cast<const bf16x8*>(b + ao[ks] + i * 16 * kRowB);
#pragma unroll
            for (int i = 0; i < T::kMT; ++i)
#pragma unroll
                for (int j = 0; j < T::kNT; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[i], bv[j], acc[i][j], 0, 0, 0);
        }
    }
    // Outputs, half of the tile's rows at a time (the waves of one wm).
    const bool isz = n0 >= p.C;
    const int width = isz ? p.Z : p.C, col0 = isz ? n0 - p.C : n0;
    uint16_t* out = isz ? p.z : p.x;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        lds_barrier();
        if ((w & 1) == half) {
#pragma unroll
            for (int i = 0; i < T::kMT; ++i)
#pragma unroll
                for (int j = 0; j < T::kNT; ++j)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        *reinterpret_cast<uint16_t*>(lds + (16 * i + 4 * lg + r) * T::kOutRow + 2 * (wn + 16 * j + li)) =
                            f32_to_bf16(acc[i][j][r]);
        }
        lds_barrier();
        constexpr int kPerRow = BN / 8, kRows = T::kThreads / kPerRow;
#pragma unroll
        for (int i = 0; i < BM / 2 / kRows; ++i) {
            const int r = i * kRows + tid / kPerRow, cc = tid % kPerRow, row = m0 + half * (BM / 2) + r;
            const u32x4 v = *reinterpret_cast<const u32x4*>(lds + r * T::kOutRow + 16 * cc);
            if (row < p.B) *reinterpret_cast<u32x4*>(out + (size_t)row * width + col0 + 8 * cc) = v;
        }
    }
}

template <int BM, int BN>
void launch_tiles(const InProj& p, int cols, hipStream_t s) {
    const int mt = (p.B + BM - 1) / BM, nt = cols / BN;
    const dim3 grid(8u * (unsigned)((mt * nt + 7) / 8)), block(Tile<BM, BN>::kThreads);
    hipLaunchKernelGGL((in_proj_tile_kernel<BM, BN>), grid, block, 0, s, p, mt, nt);
}

// Columns that a tile kernel has been launched for (0: none). The bf16 pieces only, 16-byte row
// segments, tiles not across the x | z boundary; and where the tiles cost less than 64 x 64 ones for the
// whole product. Prices in us at K = 2048 on 256 CUs (they scale with K; 8 us of the tiles' stay
// the same: the launch for the remaining columns), as measured for 100 to 4096 rows, N = 3,088 to
// 12,352 and K = 1024 to 2048: 0.048 per 64 x 64 tile (4096 rows, N = 12,352: 513 us); two 128 x 128 tiles per CU in
// 39, one in 26 (512 rows: 50 us against 70; 2048 rows: 128); a 256 x 256 tile per CU in 58 (4096 rows:
// 202 to 207 us with the launch for the remaining columns, 1,000 to 1,023 TFLOP/s, against 242 with 128 x 128).
int tile_columns(const InProj& p, hipStream_t s) {
    auto on16 = [](const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
    if (p.y || !on16(p.x) || !on16(p.z)) return 0;
    const long long cu = device_cu_count(s), all = p.C + p.Z;
    auto tiles = [&](long long cols, int t) { return ((p.B + t - 1) / t) * (cols / t); };
    const double k = p.K / 2048.0;
    const long long w128 = tiles(all, 128), half = (w128 + cu - 1) / cu;       // rounds of one tile per CU
    const double c64 = 0.048 * 256 / cu * ((p.B + 63) / 64) * ((p.N + 63) / 64);
    const double c128 = 39.0 * (half / 2) + 26.0 * (half & 1);
    const double c256 = p.C % 256 ? 1e30 : 58.0 * ((tiles(all, 256) + cu - 1) / cu);
    if (k * c64 <= 8.0 + k * std::min(c128, c256)) return 0;
    if (c256 < c128) {
        launch_tiles<256, 256>(p, (int)(all / 256 * 256), s);
        return (int)(all / 256 * 256);
    }
    launch_tiles<128, 128>(p, (int)all, s);
    return (int)all;
}

}  // namespace
}  // namespace ixg

extern "C" hipError_t ix_gdn_check_cfg_(const ix_gdn_cfg* c);

extern "C" int ix_gdn_in_proj_width(const ix_gdn_cfg* cfg) {
    if (ix_gdn_check_cfg_(cfg) != hipSuccess) return 0;
    return 2 * cfg->h_k * cfg->d_k + cfg->h_v * cfg->d_v + cfg->h_v * cfg->d_v + 2 * cfg->h_v;
}

extern "C" hipError_t ix_gdn_in_proj(const ix_gdn_cfg* cfg, int B, int hidden, const uint16_t* h, const uint16_t* w,
                                     uint16_t* x, uint16_t* z, uint16_t* a, uint16_t* b, float* y, hipStream_t s) {
    using namespace ixg;
    const hipError_t e = ix_gdn_check_cfg_(cfg);
    if (e != hipSuccess) return e;
    if (B <= 0 || B > 65535 * kMt || hidden <= 0 || hidden % kKd != 0) return hipErrorInvalidValue;
    if (!h || !w || !x || !z || !a || !b) return hipErrorInvalidValue;
    if ((reinterpret_cast<uintptr_t>(h) | reinterpret_cast<uintptr_t>(w)) & 15) return hipErrorInvalidValue;
    if (((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(z) | reinterpret_cast<uintptr_t>(a) |
          reinterpret_cast<uintptr_t>(b)) & 1) || (reinterpret_cast<uintptr_t>(y) & 3))
        return hipErrorInvalidValue;
    InProj p;
    p.h = h; p.w = w; p.x = x; p.z = z; p.a = a; p.b = b; p.y = y;
    p.B = B; p.K = hidden;
    p.C = 2 * cfg->h_k * cfg->d_k + cfg->h_v * cfg->d_v;
    p.Z = cfg->h_v * cfg->d_v;
    p.hv = cfg->h_v;
    p.N = p.C + p.Z + 2 * p.hv;
    p.n0 = tile_columns(p, s);
    const dim3 grid((unsigned)((p.N - p.n0 + kNt - 1) / kNt), (unsigned)((B + kMt - 1) / kMt));
    hipLaunchKernelGGL(in_proj_kernel, grid, dim3((kCons + kProd) * kWave), 0, s, p);
    return hipGetLastError();
}

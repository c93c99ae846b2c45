// gdn_prefill_seq.hip -- prefill with one workgroup per (sequence, one or two v heads of a q/k
// head), for gfx950.
//
// The math of gdn_prefill.hip (chunks of 64 tokens, T-form), for batches with enough sequences to
// fill the GPU: a workgroup walks its sequence's chunks with the whole 128 x 128 states of its
// heads in registers and keeps everything a chunk needs in LDS, so nothing goes through a
// workspace and no launch separates the chunk-local work from the recurrence.
//
// Columns of the state are independent: with two heads (NH = 2) waves 0-3 own head 0 and waves 4-7
// head 1, 32 columns (NT = 2 tiles) each; with one head each of the 8 waves owns 16 columns. A
// wave carries its columns from the state through D to the outputs, so no product crosses
// waves, and every A operand read from LDS serves all its tiles. Per chunk, with S the state at
// its start and the notation of gdn_prefill.hip, in four phases that end at a barrier:
//   1. conv, activation and L2 norm of the q rows (waves 0-3) and k rows (waves 4-7) into
//      split-bf16 planes; the heads' decay scans (waves 0 and 5, or wave 0);
//   2. waves 0-3: the 10 + 10 lower-triangle blocks of K K^T and Q K^T in six tasks (block_row), with
//      the heads' decays (A, M); the four 16 x 16 diagonal blocks of T = (I + A)^-1 by substitution in fp32,
//      each in the wave whose task formed it (tasks 1, 3, 4, 5: waves 1, 3, 0 and 2). All waves: W = K S
//      and Q S of their columns. Waves 4-7: the previous chunk's outputs leave LDS, a row per half wave
//      (whole 512-byte lines; the gated norm of a row sits in one half wave);
//   3. into the query planes' space: A's blocks of rows 2 and 3 left of the diagonal blocks' 32 columns
//      (waves 0 and 2), T_10 and T_32 (waves 3 and 1); V (conv of the wave's v channels) and X =
//      diag(beta) (V - diag(Gam) W);
//   4. D in two steps of 32 rows, D_b = [T_00 0; T_10 T_11] X_b of the step's diagonal block, the second on
//      X less the A blocks' product with the first (the blocks of T left of those are never formed);
//      O = diag(Gam) Q S + M D into LDS; S' = gam S + K^T diag(E) D.
// Products are split-bf16 MFMA as in gdn_prefill.hip, accumulator tiles feeding the next product
// as B operands (kperm order).
//
// What bounds it: vector instructions and the latency of the dependent phases. With SiLU and output gate
// a chunk of two heads takes 52,800 cycles on a CU (phases 1 to 4: 10.6, 23.7, 7.6 and 10.9 thousand; plain
// 6.3, 15.1, 3.5 and 11.1, in all 36,000); it issues 36,400 vector and matrix instructions of a wave, 9,100 on each
// SIMD at 4 cycles or more, and keeps a SIMD's matrix unit busy for 12,800 cycles. Workgroups of one
// head with 16 columns a wave, two per CU, repeat the q/k work for each head and spill: 967 us against 700
// (an earlier form, 32 sequences of U[1, 2048] tokens, 16 q/k, 32 v heads, gated). Products and vector
// work share a phase where waves w and w + 4 (one SIMD) can take them in opposite order; operands of the
// long product loops are read one step ahead. That batch with SiLU: 845-857 us, in windows 1,744.
#include "gdn_prefill_seq.h"

namespace ixg {
namespace {

constexpr int kSeqWaves = kSeqThreads / kWave;
// LDS (bytes): key planes; query planes, then A and the waves' v inputs in the same place; per head
// M, the diagonal blocks of T, and G, beta, exp(G), exp(G_last - G); the outputs, 64 rows of 128
// floats per head. All of a CU's 160 KiB with two heads.
constexpr int kOffK = 0, kOffR = kKSlot, kOffH = 2 * kKSlot;
// A head's blocks: A fragments (2, 0), (3, 0) (split, 2 KiB each), then T's blocks (1, 0) and (3, 2);
// in its own space M's fragments and T's diagonal blocks. T's blocks are fp32, 16 rows of 16.
constexpr int kTTile = 16 * 16 * 4, kTRow = 16 * 4, kAFrag = 2 * 1024, kABytes = 2 * kAFrag + 2 * kTTile;
constexpr int kMFragBytes = 10 * 1024, kDecBytes = 4 * kChunk * 4;
constexpr int kHeadBytes = kMFragBytes + 4 * kTTile + kDecBytes;
constexpr int kXRows = 40;                                // v inputs of 37 tokens per wave and half chunk
constexpr int kOBytes = kChunk * kD * 4;
template <int NH> struct SeqLds {
    static constexpr int kX = kOffR + NH * kABytes, kXWave = kXRows * 32 * NH;
    static constexpr int kO = kOffH + NH * kHeadBytes, kBytes = kO + NH * kOBytes;
    static_assert(kX + kSeqWaves * kXWave <= kOffH, "A and the v inputs fit the query planes");
    static_assert(kBytes <= 160 * 1024, "LDS of a CU");
};

typedef __attribute__((address_space(3))) float lds_f32;
typedef __attribute__((address_space(3))) uint32_t lds_u32;
typedef __attribute__((address_space(3))) uint16_t lds_u16;
typedef uint32_t u2x __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) u2x lds_u2x;
typedef __attribute__((address_space(3))) u4x lds_u4x;

// Task t forms the blocks (br, bc), (br, bc + 1) of the lower block triangle of both products (4 and
// 5 the first only), so that K's rows of block bc serve both and a fragment of M or A is whole in
// one wave: (3, 0) (3, 1); (3, 2) (3, 3); (2, 0) (2, 1); (1, 0) (1, 1); (2, 2); (0, 0). Waves 0-3
// take tasks 0-3, waves 0 and 2 (whose first ones hold no diagonal block to invert) also 4 and 5.
__device__ __forceinline__ int block_row(int t) { return t < 2 ? 3 : t == 2 || t == 4 ? 2 : t == 3 ? 1 : 0; }
__device__ __forceinline__ int block_col(int t) { return t == 1 || t == 4 ? 2 : 0; }

__device__ __forceinline__ bf8 pair(const bf4& a, const bf4& b) {
    return __builtin_bit_cast(bf8, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}
// acc[n][mt] += A B_n over the wave's column tiles.
template <int NT, int M>
__device__ __forceinline__ void mfma_tiles(const bf8& ah, const bf8& al, const bf8 (&bh)[NT], const bf8 (&bl)[NT],
                                           v4 (&acc)[NT][M], int mt) {
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[n][mt] = mfma_bf16(ah, bh[n], acc[n][mt]);
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[n][mt] = mfma_bf16(ah, bl[n], acc[n][mt]);
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[n][mt] = mfma_bf16(al, bh[n], acc[n][mt]);
}
__device__ __forceinline__ Split4 lds_half(const lds_u8* hi, const lds_u8* lo) {
    return Split4{__builtin_bit_cast(bf4, *(const lds_u2x*)hi), __builtin_bit_cast(bf4, *(const lds_u2x*)lo)};
}

// The wave's v inputs of one chunk, 16 NT channels: x rows -3 .. 68 of the chunk, 9 loads of 8
// rows, lane l holding 2 NT channels from 2 NT (l & 7) on of row (l >> 3) + 8 i - 3; rows past the
// sequence end repeat its last token.
template <int NT>
struct VIn {
    uint32_t w[9][NT];
};
// A row's address is a uniform base plus a 32-bit lane offset (by_sequence's rule bounds it).
__device__ __forceinline__ const char* row_at(const PrefillParams& p, int t) {
    return reinterpret_cast<const char*>(p.x) + (size_t)t * p.L.C * 2;
}
template <int NT>
__device__ __forceinline__ void v_load(const PrefillParams& p, const ChunkGeo& g, int last, int ch0, int lane, int i,
                                       VIn<NT>& v) {
    const int first = max(g.pos0 - 3, 0), rel = g.pos0 - 3 - first + (lane >> 3), most = last - first;
    const uint32_t r = (uint32_t)max(min(rel + 8 * i, most), 0);
    const uint32_t* src = reinterpret_cast<const uint32_t*>(
        row_at(p, g.lo + first) + (__umul24(r, 2 * p.L.C) + 2 * (ch0 + 2 * NT * (lane & 7))));
    if constexpr (NT == 1) {
        v.w[i][0] = src[0];
    } else {                                                 // 4-byte aligned
        typedef uint32_t u2a __attribute__((ext_vector_type(2), aligned(4)));
        const u2a x = *reinterpret_cast<const u2a*>(src);
        v.w[i][0] = x.x;
        v.w[i][1] = x.y;
    }
}
// The history in place of the rows before the sequence start (of its first chunk).
template <int DC, int NT>
__device__ __forceinline__ void v_history(const PrefillParams& p, int s, int ch0, int lane, VIn<NT>& v) {
    const uint16_t* hist = p.conv_state + (size_t)s * p.L.C * (DC - 1) + (ch0 + 2 * NT * (lane & 7)) * (DC - 1) +
                           max((lane >> 3) - 3 + DC - 1, 0);
    if (lane < 24) {
#pragma unroll
        for (int n = 0; n < NT; ++n)
            v.w[0][n] = hist[2 * n * (DC - 1)] | ((uint32_t)hist[(2 * n + 1) * (DC - 1)] << 16);
    }
}

// conv_load (gdn_chunk.h) with uniform bases and 32-bit lane offsets, in parts that a caller issues
// between other work: the DC - 1 tokens before the rows and the weights of channels ch, ch + 1,
// then two of the tokens tb .. tb + 15 of the chunk (past its end its last token repeated) at a
// time. Every workgroup reaches its loads at about the same time: issued together they would
// queue for the memory and hold up the wave.
template <int DC>
__device__ __forceinline__ void row_load_first(const PrefillParams& p, const ChunkGeo& g, int ch, int tb, ConvIn<DC>& in) {
    const Layer& L = p.L;
    uint32_t off = 2 * ch;
    __asm__ volatile("" : "+v"(off));                        // derived offsets formed here, not held
    const char* cs = reinterpret_cast<const char*>(p.conv_state) + (size_t)g.s * L.C * (DC - 1) * 2;
#pragma unroll
    for (int i = 0; i < DC - 1; ++i) {                       // the choice is uniform
        const int pos = min(g.pos0 + tb - (DC - 1) + i, g.pos0 + g.len - 1);
        const char* b = pos >= 0 ? row_at(p, g.lo + pos) : cs + 2 * (DC - 1 + pos);
        uint32_t o0 = pos >= 0 ? off : off * (DC - 1), o1 = o0 + (pos >= 0 ? 2 : 2 * (DC - 1));
        __asm__ volatile("" : "+v"(o0));
        __asm__ volatile("" : "+v"(o1));
        in.h0[i] = *reinterpret_cast<const uint16_t*>(b + o0);
        in.h1[i] = *reinterpret_cast<const uint16_t*>(b + o1);
    }
    uint32_t ow = off * DC;
    __asm__ volatile("" : "+v"(ow));
    const uint32_t* wp = reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(L.conv_w) + ow);
#pragma unroll
    for (int i = 0; i < DC; ++i) in.w[i] = wp[i];
}
template <int DC>
__device__ __forceinline__ void row_load_pair(const PrefillParams& p, const ChunkGeo& g, int ch, int tb, int i, ConvIn<DC>& in) {
    const char* base = row_at(p, g.t0);
#pragma unroll
    for (int t = 2 * i; t < 2 * i + 2; ++t) {
        uint32_t o = 2 * ch + (uint32_t)(min(tb + t, g.len - 1) * 2 * p.L.C);
        __asm__ volatile("" : "+v"(o));                      // one base, not one per row
        in.xs[t] = *reinterpret_cast<const uint32_t*>(base + o);
    }
}

// The kernel's arguments, read again: what a part of the loop needs of them, it loads where it needs
// it, instead of all of them being held in scalar registers through the loop.
struct SeqArgs {
    PrefillParams p;
    OutGate gate;
    int parts;
};
__device__ __forceinline__ SeqArgs args_again() {
    typedef const __attribute__((address_space(4))) void* kptr;
    kptr k = (kptr)__builtin_amdgcn_kernarg_segment_ptr();
    __asm__ volatile("" : "+s"(k));
    return *(const SeqArgs*)k;
}

template <int DC, bool SILU, bool GATED, int NH>
__global__ void __launch_bounds__(kSeqThreads) seq_kernel(const SeqArgs args) {
    using LdsOf = SeqLds<NH>;
    constexpr int NT = NH;
    __shared__ __align__(16) uint8_t lds[LdsOf::kBytes];
    const PrefillParams& p = args.p;
    const Layer& L = p.L;
    const int parts = args.parts;
    // Items in order of length (longest sequence first); a sequence's q/k heads side by side, the
    // parts of one q/k head h_k apart (the same XCD, whose L2 then serves their common rows).
    const int per = L.h_k * parts, rank = blockIdx.x / per, slot = blockIdx.x % per;
    const int s = p.ws.order[rank];
    if (p.ws.chunk_off[s + 1] != p.ws.chunk_off[s]) return;  // the windowed path's sequence
    const int src = slot % L.h_k, m0 = NH * (slot / L.h_k), nmap = mapped_count(L, src);
    if (m0 >= nmap) return;
    int lo, hi;
    seq_bounds(p, s, lo, hi);
    lo = __builtin_amdgcn_readfirstlane(lo);
    hi = __builtin_amdgcn_readfirstlane(hi);
    if (hi <= lo) return;
    const int tid = threadIdx.x, lane0 = tid & (kWave - 1);
    int w = __builtin_amdgcn_readfirstlane(tid / kWave);
    // This wave's head; past the last one (an odd count's second half) the waves repeat the last
    // head and store nothing.
    const int h = mapped_head(L, src, min(m0 + (NH == 2 ? w >> 2 : 0), nmap - 1));
    int hd, col0, tb;                                        // head slot, first column, first row of phase 1
    bool isk, scans;                                         // k rows; runs its head's decay scan
    auto of_wave = [&]() {
        hd = NH == 2 ? w >> 2 : 0;
        col0 = NH == 2 ? 32 * (w & 3) : 16 * w;
        tb = kConvTok * (w & 3);
        isk = w >= 4;
        scans = w == 0 || (NH == 2 && w == 5);
    };
    of_wave();
    lds_u8* ld = (lds_u8*)lds;
    auto dec_of = [&](int head, int i) {
        return (lds_f32*)(ld + kOffH + head * kHeadBytes + kMFragBytes + 4 * kTTile) + i * kChunk;
    };

    v4 S[NT][8];
    {
        const float* sl = p.state + (((size_t)s * L.h_v + h) * kD + col0) * kD + (lane0 & 15) * kD + 4 * (lane0 >> 4);
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int mt = 0; mt < 8; ++mt) S[n][mt] = *reinterpret_cast<const v4*>(sl + n * 16 * kD + 16 * mt);
    }

    const int qkch0 = isk ? k_channel(L, src, 0) : q_channel(L, src, 0);
    uint32_t cw[NT][(DC + 1) / 2];                           // conv weights of the lane's v channels, bf16 pairs
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        const uint16_t* wp = L.conv_w + (size_t)v_channel(L, h, col0 + 16 * n + (lane0 & 15)) * DC;
#pragma unroll
        for (int i = 0; i < (DC + 1) / 2; ++i)
            cw[n][i] = wp[2 * i] | (2 * i + 1 < DC ? (uint32_t)wp[2 * i + 1] << 16 : 0u);
    }

    ChunkGeo g;
    g.s = s;
    g.lo = lo;
    auto geo = [&](int t0) {
        g.t0 = t0;
        g.len = min(kChunk, hi - t0);
        g.pos0 = t0 - lo;
    };
    ConvIn<DC> in;
    // The outputs of the chunk at t0 from LDS: a row per half wave, 4 columns per lane; wave w of 4-7
    // takes rows 16 (w - 4) .. + 15 of every head. A row's 16-column groups are XOR-swizzled by its
    // row quad.
    constexpr int R = 4;                                     // of 8 pairs of rows, two groups
    auto head_of = [&](const Layer& L, int e) { return mapped_head(L, src, min(m0 + e, nmap - 1)); };
    auto out_at = [&](int e, int row, int col) {
        return (lds_f32*)(ld + LdsOf::kO + e * kOBytes) + row * kD + (col ^ (16 * ((row >> 2) & 3)));
    };
    auto load_z = [&](int e, int i0, int t0, int len, int lane, uint2 (&z)[R]) {
        const SeqArgs again = args_again();
        const int hv = again.p.L.h_v;
        const uint16_t* zb = again.gate.z + ((size_t)t0 * hv + head_of(again.p.L, e)) * kD;
#pragma unroll
        for (int i = 0; i < R; ++i)
            z[i] = *reinterpret_cast<const uint2*>(
                zb + ((uint32_t)min(16 * (w - 4) + (lane >> 5) + 2 * (i0 + i), len - 1) * hv * kD + 4 * (lane & 31)));
    };
    // Row pairs i0 .. i0 + R - 1 of head e.
    auto out_rows = [&](int e, int i0, const uint2 (&z)[R], int t0, int len, int lane) {
        const SeqArgs again = args_again();
        const PrefillParams& p = again.p;
        const OutGate& gate = again.gate;
        // The rows of an output that exist, as a buffer: stores past them (or of the repeated head past
        // an odd count) are dropped by the bounds check.
        const uint32_t ostep = (uint32_t)p.L.h_v * kD;
        const size_t base = ((size_t)t0 * p.L.h_v + head_of(p.L, e)) * kD;
        const bool live = m0 + e < nmap;
        auto rows_of = [&](void* out, int bytes) {
            return __builtin_amdgcn_make_buffer_rsrc(static_cast<char*>(out) + base * bytes, 0,
                                                     live ? (int)(((uint32_t)(len - 1) * ostep + kD) * bytes) : 0, 0x00020000);
        };
        const int r0 = 16 * (w - 4) + (lane >> 5) + 2 * i0, oc = 4 * (lane & 31);
        const uint32_t at = (uint32_t)r0 * ostep + oc;
        v4 nrm;
        if constexpr (GATED) {
            nrm = *reinterpret_cast<const v4*>(gate.nrm + oc);
            // q8_1 blocks from the same values, formed for themselves: kept apart and rolled up, their
            // divisions would otherwise be most of the loop's code. Ahead of the stores: y_bf16 may overwrite z.
            if (gate.y_q8_1) {
#pragma clang loop unroll(disable)
                for (int i = 0; i < R; ++i) {
                    const int row = r0 + 2 * i;
                    const uint32_t ra = (uint32_t)min(row, len - 1) * ostep + oc;
                    const v4 v = *(const lds_v4*)out_at(e, row, oc);
                    const v4 y = gate_row4(gate, v, nrm, *reinterpret_cast<const uint2*>(gate.z + base + ra));
                    q81_store4(y, lane, live && row < len ? gate.y_q8_1 + (base + ra) / 32 * kQ81Bytes : nullptr);
                }
            }
        }
        v4 o[R];
#pragma unroll
        for (int i = 0; i < R; ++i) o[i] = *(const lds_v4*)out_at(e, r0 + 2 * i, oc);
        auto store32 = [&](float* out) {
            const auto b = rows_of(out, 4);
#pragma unroll
            for (int i = 0; i < R; ++i)
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4x, o[i]), b, (at + 2 * i * ostep) * 4, 0, 0);
        };
        auto store16 = [&](uint16_t* out) {
            const auto b = rows_of(out, 2);
#pragma unroll
            for (int i = 0; i < R; ++i)
                __builtin_amdgcn_raw_buffer_store_b64(u2x{pack_bf16x2(o[i][0], o[i][1]), pack_bf16x2(o[i][2], o[i][3])}, b,
                                                      (at + 2 * i * ostep) * 2, 0, 0);
        };
        if (p.o) store32(p.o);
        if (p.o_bf16) store16(p.o_bf16);
        if constexpr (GATED) {
#pragma unroll
            for (int i = 0; i < R; ++i) o[i] = gate_row4(gate, o[i], nrm, z[i]);
            if (gate.y) store32(gate.y);
            if (gate.y_bf16) store16(gate.y_bf16);
        }
    };

    geo(lo);
    row_load_first<DC>(p, g, qkch0 + 2 * lane0, tb, in);
#pragma unroll
    for (int i = 0; i < kConvTok / 2; ++i) row_load_pair<DC>(p, g, qkch0 + 2 * lane0, tb, i, in);
    VIn<NT> vin;
    const int vch = v_channel(L, h, col0);
#pragma unroll
    for (int i = 0; i < 9; ++i) v_load<NT>(p, g, hi - lo - 1, vch, lane0, i, vin);
    v_history<DC, NT>(p, s, vch, lane0, vin);
    for (int t0 = lo;; t0 += kChunk) {
        const int len = g.len;
        // The lane index, made opaque at the start of each phase: a phase then derives its addresses
        // from it where it uses them, instead of holding every phase's through the whole loop.
        int lane = lane0, li, lg4;
        auto phase = [&]() {
            __asm__ volatile("" : "+v"(lane), "+s"(w));
            li = lane & 15;
            lg4 = lane >> 4;
            of_wave();
        };
        phase();
        const bool main = t0 < hi;                           // false once more, for the last outputs
        u2x uh[NH][2] = {}, ul[NH][2] = {};
        if (main) {
            // 1. q and k rows; the gate inputs of the scanning waves, loaded ahead of them (lane = token)
            uint16_t ra = 0, rb = 0;
            float A_log = 0.0f, dt_bias = 0.0f;
            if (scans) {
                const SeqArgs again = args_again();
                const size_t ab = (size_t)(t0 + min(lane, len - 1)) * again.p.L.h_v + h;
                ra = again.p.a[ab];
                rb = again.p.b[ab];
                A_log = again.p.L.A_log[h];
                dt_bias = again.p.L.dt_bias[h];
            }
            {
                // Channel pair (2 l, 2 l + 1) of a plane row: channel 32 b + 16 u + 4 a + e sits in
                // chunk 4 b + a at entry 4 u + e.
                const int c2 = 2 * lane, cj = 16 * (4 * (c2 >> 5) + ((c2 >> 2) & 3)), ce = 2 * (4 * ((c2 >> 4) & 1) + (c2 & 3));
                const int nt = min(max(len - tb, 0), kConvTok);
                float y0[kConvTok], y1[kConvTok];
                conv_run<DC, SILU, true>(in, y0, y1);
                float ss[kConvTok];
#pragma unroll
                for (int t = 0; t < kConvTok; ++t) ss[t] = fmaf(y0[t], y0[t], y1[t] * y1[t]);
                const SeqArgs again = args_again();
                const float scale = isk ? 1.0f : again.p.L.q_scale;
                const float inv_l = scale * rsqrtf(sum16_scatter(ss, lane) + again.p.L.l2_eps);
                lds_u8* dst = ld + (isk ? kOffK : kOffR) + tb * kPRow + ce;
#pragma unroll
                for (int t = 0; t < kConvTok; ++t) {
                    const float inv = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(inv_l), 4 * t));
                    uint32_t vh = 0, vl = 0;
                    if (t < nt) split2(y0[t] * inv, y1[t] * inv, vh, vl);
                    lds_u8* d = dst + (cj ^ (16 * kswz(t))) + t * kPRow;
                    *(lds_u32*)d = vh;
                    *(lds_u32*)(d + kKPlane) = vl;
                }
            }
            if (scans) {                                         // lane = token
                const bool ok = lane < len;
                float lg = ok ? log_gate(A_log, dt_bias, bf16_to_f32(ra)) : 0.0f;
                lg = wave_scan(lg);
                const float last = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(lg), kChunk - 1));
                dec_of(hd, 0)[lane] = lg;
                dec_of(hd, 1)[lane] = ok ? sigmoid_f(bf16_to_f32(rb)) : 0.0f;
                dec_of(hd, 2)[lane] = expf(lg);
                dec_of(hd, 3)[lane] = expf(last - lg);
            }
            lds_barrier();

            phase();
            // 2. blocks of K K^T and Q K^T, transposed (lane (li, lg4) holds t = 16 br + li, s = 16 bc +
            // 4 lg4 + r), with each head's decays: M split into its fragments, the diagonal blocks of
            // A (tasks 1, 3, 4, 5) in fp32 and inverted, the others held until the query planes are free
            if (w < 4) {
#pragma clang loop unroll(disable)
                for (int task = w; task < 6; task = task < 4 && !(w & 1) ? 4 + (w >> 1) : 6) {
                    const int br = block_row(task), bc = block_col(task);
                    v4 kk[2], qk[2];
#pragma unroll
                    for (int j = 0; j < 2; ++j) kk[j] = qk[j] = v4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int ks = 0; ks < 4; ++ks) {
                        const lds_u8* kb = ld + kOffK + k_lane(li, lg4, ks);
                        bf8 bh, bl, qh, ql, ah, al;
                        k_frag(kb + br * 16 * kPRow, 0, bh, bl);
                        k_frag(kb + (kOffR - kOffK) + br * 16 * kPRow, 0, qh, ql);
#pragma unroll
                        for (int j = 0; j < 2; ++j) {
                            k_frag(kb + min(bc + j, 3) * 16 * kPRow, 0, ah, al);
                            kk[j] = mfma_split(ah, al, bh, bl, kk[j]);
                            qk[j] = mfma_split(ah, al, qh, ql, qk[j]);
                        }
                    }
                    const int t = 16 * br + li;
                    const bool dg = task == 1 || task >= 3;          // one of its blocks is a diagonal one
#pragma unroll
                    for (int e = 0; e < NH; ++e) {
                        lds_f32* const G = dec_of(e, 0);
                        const float gt = G[t], bt = dec_of(e, 1)[t];
                        lds_u8* eb = ld + kOffH + e * kHeadBytes;
                        u2x mh[2], ml[2];
                        v4 diag = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                        for (int j = 0; j < 2; ++j) {
                            const int s0 = 16 * min(bc + j, 3) + 4 * lg4;
                            const v4 gs = *(const lds_v4*)(G + s0);
                            v4 m, a;
#pragma unroll
                            for (int r = 0; r < 4; ++r) {
                                const float d = __expf(fminf(gt - gs[r], 0.0f));
                                m[r] = s0 + r <= t ? d * qk[j][r] : 0.0f;
                                a[r] = s0 + r < t ? bt * d * kk[j][r] : 0.0f;
                            }
                            uint32_t h0, h1, l0, l1;
                            split2(m[0], m[1], h0, l0);
                            split2(m[2], m[3], h1, l1);
                            mh[j] = u2x{h0, h1};
                            ml[j] = u2x{l0, l1};
                            if (j == (task < 4)) diag = a;           // task 1's and 3's second, 4's and 5's first
                            split2(-a[0], -a[1], h0, l0);
                            split2(-a[2], -a[3], h1, l1);
                            if (task < 4) {
                                uh[e][j] = u2x{h0, h1};
                                ul[e][j] = u2x{l0, l1};
                            }
                        }
                        lds_u8* d = eb + tri_frag_at(br, bc >> 1, 0, lane);
                        if (task < 4) {
                            *(lds_u4x*)d = u4x{mh[0].x, mh[0].y, mh[1].x, mh[1].y};
                            *(lds_u4x*)(d + 1024) = u4x{ml[0].x, ml[0].y, ml[1].x, ml[1].y};
                        } else {
                            *(lds_u2x*)d = mh[0];
                            *(lds_u2x*)(d + 512) = ml[0];
                        }
                        if (dg) *(lds_v4*)(eb + kMFragBytes + br * kTTile + li * kTRow + 16 * lg4) = diag;
                    }
                    // T's diagonal block by substitution, lane = 16 head + column: row by row, the next row
                    // read while one is summed.
                    if (dg && lane < 16 * NH) {
                        wave_lds_sync();
                        lds_u8* tt = ld + kOffH + lg4 * kHeadBytes + kMFragBytes + br * kTTile;
                        float x[16];
                        v4 nx[4];
                        nx[0] = *(const lds_v4*)(tt + kTRow);
#pragma unroll
                        for (int r = 0; r < 16; ++r) {
                            v4 av[4];
#pragma unroll
                            for (int q4 = 0; q4 < 4; ++q4) {
                                if (4 * q4 < r) av[q4] = nx[q4];
                                if (r > 0 && 4 * q4 < r + 1 && r < 15) nx[q4] = *(const lds_v4*)(tt + (r + 1) * kTRow + q4 * 16);
                            }
                            float acc = r == li ? 1.0f : 0.0f;
#pragma unroll
                            for (int q = 0; q < r; ++q) acc = fmaf(-av[q >> 2][q & 3], x[q], acc);
                            x[r] = acc;
                            __builtin_amdgcn_sched_barrier(0);
                        }
                        __asm__ volatile("" ::: "memory");
#pragma unroll
                        for (int r = 0; r < 16; ++r) *(lds_f32*)(tt + r * kTRow + li * 4) = x[r];
                    }
                }
            }
        }
        // W = K S and Q S of the wave's columns; then, in waves 4-7, the previous chunk's outputs. (Waves
        // w and w + 4 share a SIMD: one's vector work runs beside the other's products.)
        v4 W[NT][4], O[NT][4];
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int mt = 0; mt < 4; ++mt) W[n][mt] = O[n][mt] = v4{0.f, 0.f, 0.f, 0.f};
        if (main) {
            phase();
            // 32 steps (ks, mt, K or Q), the next step's operand read while one multiplies
            bf8 f[2][2], sh[NT], sl[NT];
            auto operand = [&](int i, bf8 (&x)[2]) {
                k_frag(ld + (i & 1 ? kOffR : kOffK) + k_lane(li, lg4, i >> 3), (i >> 1) & 3, x[0], x[1]);
            };
            operand(0, f[0]);
#pragma unroll
            for (int i = 0; i < 32; ++i) {
                const int ks = i >> 3, mt = (i >> 1) & 3;
                if ((i & 7) == 0) {
#pragma unroll
                    for (int n = 0; n < NT; ++n) split_tiles(S[n][2 * ks], S[n][2 * ks + 1], sh[n], sl[n]);
                }
                if (i < 31) operand(i + 1, f[(i + 1) & 1]);
                mfma_tiles<NT>(f[i & 1][0], f[i & 1][1], sh, sl, i & 1 ? O : W, mt);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        phase();
        if (w >= 4 && t0 > lo) {
            const int tp = t0 - kChunk, lp = min(kChunk, hi - tp);
            uint2 z[2][R];                                   // the gate's inputs of a group, the next one's ahead
            if constexpr (GATED) load_z(0, 0, tp, lp, lane, z[0]);
#pragma unroll
            for (int i = 0; i < 2 * NH; ++i) {
                if constexpr (GATED)
                    if (i + 1 < 2 * NH) load_z((i + 1) >> 1, R * ((i + 1) & 1), tp, lp, lane, z[(i + 1) & 1]);
                out_rows(i >> 1, R * (i & 1), z[i & 1], tp, lp, lane);
            }
        }
        if (!main) break;
        lds_barrier();

        phase();
        // 3. A over the query planes; T_10 = -T_11 A_10 T_00 (wave 3) and T_32 (wave 1)
        if (w < 4) {
            const int br = block_row(w);
#pragma unroll
            for (int e = 0; e < NH; ++e) {
                lds_u8* ab = ld + kOffR + e * kABytes;
                if (w == 0 || w == 2) {
                    lds_u8* d = ab + (br - 2) * kAFrag + lane * 16;
                    *(lds_u4x*)d = u4x{uh[e][0].x, uh[e][0].y, uh[e][1].x, uh[e][1].y};
                    *(lds_u4x*)(d + 1024) = u4x{ul[e][0].x, ul[e][0].y, ul[e][1].x, ul[e][1].y};
                } else {
                    const lds_u8* tt = ld + kOffH + e * kHeadBytes + kMFragBytes + (br - 1) * kTTile;
                    v4 t0c;                                  // T_00 as a B operand
#pragma unroll
                    for (int r = 0; r < 4; ++r) t0c[r] = *(const lds_f32*)(tt + (4 * lg4 + r) * kTRow + 4 * li);
                    const v4 t1 = *(const lds_v4*)(tt + kTTile + li * kTRow + 16 * lg4);
                    const Split4 na{__builtin_bit_cast(bf4, uh[e][0]), __builtin_bit_cast(bf4, ul[e][0])};   // -A_10
                    const v4 zero = {0.f, 0.f, 0.f, 0.f};
                    const v4 t10 = mfma16_split(split4(t1), split4(mfma16_split(na, split4(t0c), zero)), zero);
                    lds_u8* d = ab + 2 * kAFrag + (br >> 1) * kTTile;
#pragma unroll
                    for (int r = 0; r < 4; ++r) *(lds_f32*)(d + (4 * lg4 + r) * kTRow + 4 * li) = t10[r];
                }
            }
        }
        // V and X
        {
            lds_u8* xs = ld + LdsOf::kX + w * LdsOf::kXWave;
            constexpr int kRow = 32 * NT;
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                wave_lds_sync();
                __asm__ volatile("" ::: "memory");
#pragma unroll
                for (int i = 0; i < 5; ++i) {
                    lds_u8* d = xs + (8 * i + (lane >> 3)) * kRow + 4 * NT * (lane & 7);
                    if constexpr (NT == 1) *(lds_u32*)d = vin.w[4 * half + i][0];
                    else *(lds_u2x*)d = u2x{vin.w[4 * half + i][0], vin.w[4 * half + i][NT - 1]};
                }
                wave_lds_sync();
                __asm__ volatile("" ::: "memory");
#pragma unroll
                for (int m = 0; m < 2; ++m) {
                    const int mt = 2 * half + m, tr = 16 * mt + 4 * lg4;
                    const v4 gm = *(const lds_v4*)(dec_of(hd, 2) + tr), bt = *(const lds_v4*)(dec_of(hd, 1) + tr);
#pragma unroll
                    for (int n = 0; n < NT; ++n) {
                        float xv[DC + 3];
#pragma unroll
                        for (int j = 0; j < DC + 3; ++j)
                            xv[j] = __uint_as_float((uint32_t) * (const lds_u16*)(xs + (16 * m + 4 * lg4 + 4 - DC + j) * kRow + 32 * n + 2 * li) << 16);
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            float acc = 0.0f;
#pragma unroll
                            for (int i = 0; i < DC; ++i) acc = fmaf(xv[e + i], bf16_half(cw[n][i >> 1], i & 1), acc);
                            if constexpr (SILU) acc = acc * sigmoid_r(acc);
                            acc = tr + e < len ? acc : 0.0f;
                            W[n][mt][e] = bt[e] * fmaf(-gm[e], W[n][mt][e], acc);
                        }
                    }
                }
            }
        }
        lds_barrier();

        phase();
        // 4. D by forward substitution over the two 32-row blocks, O and S'
        {
            const lds_u8* af = ld + kOffR + hd * kABytes;
            const lds_u8* hb = ld + kOffH + hd * kHeadBytes;
            bf8 dh[2][NT], dl[2][NT];                        // D, split, 32 rows each
            bf8 eh[2][NT], el[2][NT];                        // diag(E) D
            // Row block b (0, 1): D = [T_00 0; T_10 T_11] X
            auto solve = [&](int b) {
                const lds_u8* tt = hb + kMFragBytes + 2 * b * kTTile + li * kTRow + 16 * lg4;
                const v4 t00 = *(const lds_v4*)tt, t11 = *(const lds_v4*)(tt + kTTile);
                const v4 t10 = *(const lds_v4*)(af + 2 * kAFrag + b * kTTile + li * kTRow + 16 * lg4);
                const v4 e0 = *(const lds_v4*)(dec_of(hd, 3) + 32 * b + 4 * lg4), e1 = *(const lds_v4*)(dec_of(hd, 3) + 32 * b + 16 + 4 * lg4);
                bf8 xh[NT], xl[NT], ah, al;
                v4 D[NT][2];
#pragma unroll
                for (int n = 0; n < NT; ++n) {
                    split_tiles(W[n][2 * b], W[n][2 * b + 1], xh[n], xl[n]);
                    D[n][0] = D[n][1] = v4{0.f, 0.f, 0.f, 0.f};
                }
                const Split4 s00 = split4(t00);
                mfma_tiles<NT>(pair(s00.h, bf4{0, 0, 0, 0}), pair(s00.l, bf4{0, 0, 0, 0}), xh, xl, D, 0);
                split_tiles(t10, t11, ah, al);
                mfma_tiles<NT>(ah, al, xh, xl, D, 1);
#pragma unroll
                for (int n = 0; n < NT; ++n) {
                    split_tiles(D[n][0], D[n][1], dh[b][n], dl[b][n]);
                    split_tiles(D[n][0] * e0, D[n][1] * e1, eh[b][n], el[b][n]);
                }
            };
            // (0, 0) and (2, 1) of M pair a diagonal block with a zero block.
            auto m_frag = [&](int m, int ks, bf8& mh, bf8& ml) {
                if (tri_half(m, ks)) {
                    const Split4 v = lds_half(hb + tri_frag_at(m, ks, 0, lane), hb + tri_frag_at(m, ks, 1, lane));
                    mh = pair(v.h, bf4{0, 0, 0, 0});
                    ml = pair(v.l, bf4{0, 0, 0, 0});
                } else {
                    mh = *(const lds_bf8*)(hb + tri_frag_at(m, ks, 0, lane));
                    ml = *(const lds_bf8*)(hb + tri_frag_at(m, ks, 1, lane));
                }
            };
            bf8 ah, al;
            solve(0);
#pragma unroll
            for (int m = 2; m < 4; ++m) {
                ah = *(const lds_bf8*)(af + (m - 2) * kAFrag + lane * 16);
                al = *(const lds_bf8*)(af + (m - 2) * kAFrag + 1024 + lane * 16);
                mfma_tiles<NT>(ah, al, dh[0], dl[0], W, m);
            }
#pragma unroll
            for (int mt = 0; mt < 4; ++mt) {
                const v4 gm = *(const lds_v4*)(dec_of(hd, 2) + 16 * mt + 4 * lg4);
#pragma unroll
                for (int n = 0; n < NT; ++n) O[n][mt] *= gm;
                m_frag(mt, 0, ah, al);
                mfma_tiles<NT>(ah, al, dh[0], dl[0], O, mt);
            }
            solve(1);
#pragma unroll
            for (int mt = 2; mt < 4; ++mt) {
                m_frag(mt, 1, ah, al);
                mfma_tiles<NT>(ah, al, dh[1], dl[1], O, mt);
            }
#pragma unroll
            for (int n = 0; n < NT; ++n)
#pragma unroll
                for (int mt = 0; mt < 4; ++mt)
#pragma unroll
                    for (int r = 0; r < 4; ++r) *out_at(hd, 16 * mt + 4 * lg4 + r, col0 + 16 * n + li) = O[n][mt][r];
            // S', with the next chunk's loads issued a few at a time in between: its q, k and v rows (the
            // last chunk's again at the end).
            phase();
            if (t0 + kChunk < hi) geo(t0 + kChunk);
            const SeqArgs again = args_again();
            row_load_first<DC>(again.p, g, qkch0 + 2 * lane, tb, in);
            const float gam = dec_of(hd, 2)[kChunk - 1];
            bf8 f[2][4];                                     // K^T of a row tile, the next one's read ahead
            auto operands = [&](int mt, bf8 (&x)[4]) {
                const lds_u8* kt = ld + kOffK + kt_lane(li, lg4, mt >> 1);
                kt_frag(kt, mt & 1, 0, x[0], x[1]);
                kt_frag(kt, mt & 1, 1, x[2], x[3]);
            };
            operands(0, f[0]);
#pragma unroll
            for (int mt = 0; mt < 8; ++mt) {
#pragma unroll
                for (int n = 0; n < NT; ++n) S[n][mt] *= gam;
                if (mt < 7) operands(mt + 1, f[(mt + 1) & 1]);
                const bf8(&x)[4] = f[mt & 1];
                mfma_tiles<NT>(x[0], x[1], eh[0], el[0], S, mt);
                mfma_tiles<NT>(x[2], x[3], eh[1], el[1], S, mt);
                row_load_pair<DC>(again.p, g, qkch0 + 2 * lane, tb, mt, in);
                v_load<NT>(again.p, g, hi - lo - 1, vch, lane, mt, vin);
                if (mt == 7) v_load<NT>(again.p, g, hi - lo - 1, vch, lane, 8, vin);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        lds_barrier();                                       // keys, A, T and M read for the last time
    }
    if (m0 + hd >= nmap) return;
    const SeqArgs again = args_again();
    float* const st = again.p.state + (((size_t)s * again.p.L.h_v + h) * kD + col0) * kD;
    {
        int l = lane0;
        __asm__ volatile("" : "+v"(l));
        float* sl = st + (l & 15) * kD + 4 * (l >> 4);
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int mt = 0; mt < 8; ++mt) *reinterpret_cast<v4*>(sl + n * 16 * kD + 16 * mt) = S[n][mt];
    }
    // The wave's new v histories (the old ones were read in the first chunk).
    if (lane0 < 16 * NT) {
        const int ch = v_channel(again.p.L, h, col0 + lane0);
        hist_put(again.p, ch, s, hist_fetch(again.p, ch, lo, hi - lo, s));
    }
}

// The new q/k conv histories of the sequences seq_kernel took, after all their heads have read
// the old ones: grid (n_seq, ceil(2 h_k 128 / 256)).
__global__ void __launch_bounds__(256) seq_history_kernel(const PrefillParams p) {
    const int s = blockIdx.x, ch = blockIdx.y * 256 + threadIdx.x;
    if (ch >= 2 * p.L.h_k * kD) return;
    if (p.ws.chunk_off[s + 1] != p.ws.chunk_off[s]) return;
    int lo, hi;
    seq_bounds(p, s, lo, hi);
    if (hi > lo) hist_put(p, ch, s, hist_fetch(p, ch, lo, hi - lo, s));
}

template <int DC, bool SILU, int NH>
void launch(const PrefillParams& p, const OutGate* gate, hipStream_t s) {
    const int parts = (int)(seq_workgroups(p.L) / p.L.h_k);
    const dim3 grid((unsigned)(p.n_seq * seq_workgroups(p.L))), block(kSeqThreads);
    const SeqArgs args{p, gate ? *gate : OutGate{}, parts};
    if (gate) hipLaunchKernelGGL((seq_kernel<DC, SILU, true, NH>), grid, block, 0, s, args);
    else hipLaunchKernelGGL((seq_kernel<DC, SILU, false, NH>), grid, block, 0, s, args);
}

template <int DC>
void launch(const PrefillParams& p, const OutGate* gate, bool silu, hipStream_t s) {
    const bool two = p.L.h_v > p.L.h_k;
    if (silu) two ? launch<DC, true, 2>(p, gate, s) : launch<DC, true, 1>(p, gate, s);
    else two ? launch<DC, false, 2>(p, gate, s) : launch<DC, false, 1>(p, gate, s);
}

}  // namespace

long long seq_workgroups(const Layer& L) {
    const int most = L.head_map == IX_GDN_HEAD_MOD ? (L.h_v + L.h_k - 1) / L.h_k : L.per_src, nh = L.h_v > L.h_k ? 2 : 1;
    return (long long)L.h_k * ((most + nh - 1) / nh);
}

void launch_prefill_seq(const PrefillParams& p, const OutGate* gate, bool silu, hipStream_t s) {
    switch (p.L.dc) {
        case 2: launch<2>(p, gate, silu, s); break;
        case 3: launch<3>(p, gate, silu, s); break;
        default: launch<4>(p, gate, silu, s); break;
    }
    hipLaunchKernelGGL(seq_history_kernel, dim3((unsigned)p.n_seq, (unsigned)((2 * p.L.h_k * kD + 255) / 256)), dim3(256),
                       0, s, p);
}

}  // namespace ixg

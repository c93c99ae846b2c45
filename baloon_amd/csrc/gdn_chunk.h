// gdn_chunk.h -- what the two prefill paths share (gdn_prefill.hip: chunk kernel and chain per
// window of chunks; gdn_prefill_seq.hip: one workgroup per (sequence, v head)): the launch
// parameters and workspace layout, the conv of a chunk's rows, the rolling conv history, and
// the split-bf16 key planes and fragments the MFMA products read (gfx950).
#pragma once
#include "gdn_common.h"

namespace ixg {

constexpr int kChunk = 64;

// ---------------------------------------------------------------------------------------
// Workspace layout (host and device agree through this struct)
// ---------------------------------------------------------------------------------------
// The chunk tables cover every chunk; the chunk operands cover one window of W chunks (the
// kernels run window by window, W chosen to fit the caller's workspace).
struct Ws {
    int32_t* seq_lo;     // [n_seq + 1] clamped token offsets
    int32_t* chunk_off;  // [n_seq + 1] first chunk of each sequence; chunk_off[n_seq] = #chunks
    int4* chunk_rec;     // [NC] {sequence, first token, sequence start, sequence end}
    uint8_t* Tf;         // [W][h_v] T' = (I + A)^-1 diag(beta) (64 x 64) as split-bf16 A fragments
                         // (the nonzero ones, kTriFragBytes per head)
    uint8_t* Mf;         // [W][h_v] M (64 x 64) as split-bf16 A fragments (kFragMBytes per head)
    float* G;            // [W][h_v][2][64] decay factors exp(G_last - G_t), then exp(G_t), of the
                         // inclusive cumulative log decay G (padded rows repeat the last)
    uint8_t* Kp;         // [W][h_k] normalised keys as split-bf16 planes in the chain's LDS layout
    uint16_t* Qf;        // [W][h_k] Q (64 x 128) as split-bf16 A fragments
    int32_t* order;      // [n_seq] sequences by descending length, over Tf's space: written by the
                         // plan, read before the first window writes there
};
constexpr int kWsSections = 8;
constexpr int kTriFragBytes = 10 * 1024;                // T' of one (chunk, v head)
constexpr int kFragMBytes = 16 * 1024;                  // M of one (chunk, v head)
constexpr int kPRow = 2 * 128;                          // key plane row: 128 bf16 as 16 chunks of 16 bytes
constexpr int kKPlane = 64 * kPRow;                     // one plane (hi or lo) of 64 keys
constexpr int kKSlot = 2 * kKPlane;                     // hi, then lo: 32 KiB
// Chunk j of key row t is stored at chunk j ^ kswz(t) of its row: the two 2-bit halves of
// t mod 16 swapped, so that the chain's 16-byte fragment reads (16 rows, one chunk column) and
// its transposing 8-byte reads (4 rows x 4 chunk columns per lane group) hit 16 distinct chunks.
__host__ __device__ constexpr int kswz(int t) { return ((t & 3) << 2) | ((t >> 2) & 3); }

inline size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

// Chunks of (n_seq, T) at most: each sequence adds at most one partial chunk.
inline size_t max_chunks(int n_seq, int T) { return (size_t)(T + kChunk - 1) / kChunk + (size_t)n_seq; }

// Byte offsets of every workspace section for (n_seq, T) in windows of W chunks; returns the
// total size.
inline size_t ws_layout(const ix_gdn_cfg* c, int n_seq, int T, size_t W, size_t off[kWsSections]) {
    const size_t NC = max_chunks(n_seq, T);
    const size_t sz[kWsSections] = {
        sizeof(int32_t) * (n_seq + 1), sizeof(int32_t) * (n_seq + 1), sizeof(int4) * NC,
        (size_t)kTriFragBytes * W * c->h_v, (size_t)kFragMBytes * W * c->h_v, sizeof(float) * W * c->h_v * 2 * kChunk, (size_t)kKSlot * W * c->h_k,
        sizeof(uint16_t) * W * c->h_k * 4 * 4 * 2 * 512,
    };
    size_t pos = 0;
    for (int i = 0; i < kWsSections; ++i) { off[i] = pos; pos += align256(sz[i]); }
    return pos;
}

inline Ws ws_bind(char* base, const size_t off[kWsSections]) {
    Ws w;
    w.seq_lo = reinterpret_cast<int32_t*>(base + off[0]);
    w.chunk_off = reinterpret_cast<int32_t*>(base + off[1]);
    w.chunk_rec = reinterpret_cast<int4*>(base + off[2]);
    w.Tf = reinterpret_cast<uint8_t*>(base + off[3]);
    w.Mf = reinterpret_cast<uint8_t*>(base + off[4]);
    w.G = reinterpret_cast<float*>(base + off[5]);
    w.Kp = reinterpret_cast<uint8_t*>(base + off[6]);
    w.Qf = reinterpret_cast<uint16_t*>(base + off[7]);
    w.order = reinterpret_cast<int32_t*>(base + off[3]);
    return w;
}

struct PrefillParams {
    Layer L;
    Ws ws;
    const int32_t* cu;          // [n_seq + 1]
    const uint16_t* x;          // [T][C]
    uint16_t* conv_state;       // [n_seq][C][dc-1]
    const uint16_t* a;          // [T][h_v]
    const uint16_t* b;          // [T][h_v]
    float* state;               // [n_seq][h_v][d_v][d_k]
    float* o;                   // [T][h_v][128], the window's rows (o_win), or null
    uint16_t* o_bf16;           // [T][h_v][128] or null
    int n_seq, T, NC;
    int single;                 // n_seq == 1: no plan pass; the geometry comes from cu[0], cu[1]
    int cb, W;                  // the window: chunks cb .. cb + W - 1
    int G;                      // chain workgroups per (v head, strip) in a window (1 for n_seq == 1)
    int by_seq;                 // sequences up to a length that the plan chooses go to seq_kernel
    float cost_start, cost_seq, cost_work, cost_win, cost_chain;   // its prices (us; the first once, the others per chunk)
    int o_win;                  // o holds the window's chunks only, 64 rows each
};

// Clamped bounds [lo, hi) of sequence s: the plan's seq_lo (running maximum of the offsets,
// clamped to [0, T]), or for a single sequence the same two values from cu directly.
__device__ __forceinline__ void seq_bounds(const PrefillParams& p, int s, int& lo, int& hi) {
    if (p.single) {
        lo = min(max(p.cu[0], 0), p.T);
        hi = max(min(max(p.cu[1], 0), p.T), lo);
    } else {
        lo = p.ws.seq_lo[s];
        hi = p.ws.seq_lo[s + 1];
    }
}

// Geometry of a chunk: sequence, first token, tokens in the chunk, position of the first token
// within its sequence, the sequence's first token.
struct ChunkGeo { int s, t0, len, pos0, lo; };

// ---------------------------------------------------------------------------------------
// Conv of 16 consecutive tokens of a chunk for the channel pair (ch, ch + 1), one pair per
// lane, so that every x access of a wave is one 256-byte row segment. Tokens tb .. tb + n - 1
// of the chunk (n wave-uniform, 1..16); the history of the first one comes from x or, before
// the sequence start, from the sequence's conv state ([C][dc-1] per sequence: channel ch's
// entries, then channel ch+1's).
// The loads and the arithmetic are separate steps, so that a wave can issue the loads well
// before it needs the rows (and before stores it issues in between, which its later waits
// would otherwise include).
// ---------------------------------------------------------------------------------------
constexpr int kConvTok = 16;

// The loads are unconditional and nothing touches the loaded words before conv_run: a
// load on one path only, or any use of a loaded value, makes the wave wait for every load
// it has in flight. Every row index is clamped into the chunk's tokens, so a wave whose
// rows all lie past the chunk end (n = 0) reads valid rows, whose results are discarded.
template <int DC>
struct ConvIn {
    uint32_t h0[DC - 1], h1[DC - 1];    // history of the first token (one bf16 each), oldest first
    uint32_t xs[kConvTok];              // bf16 pairs: inputs of the tokens (rows past n repeat row n-1)
    uint32_t w[DC];                     // bf16 pairs: conv weights of channel ch, then ch + 1
};

template <int DC>
__device__ __forceinline__ void conv_load(const PrefillParams& p, const ChunkGeo& g, int lo, int ch, int tb, int n,
                                          ConvIn<DC>& in) {
    const Layer& L = p.L;
#pragma unroll
    for (int i = 0; i < DC - 1; ++i) {
        const int pos = min(g.pos0 + tb - (DC - 1) + i, g.pos0 + g.len - 1);   // wave-uniform
        const uint16_t* xp = p.x + (size_t)(lo + max(pos, 0)) * L.C + ch;
        const uint16_t* sp = p.conv_state + ((size_t)g.s * L.C + ch) * (DC - 1) + (DC - 1) + min(pos, -1);
        in.h0[i] = *(pos >= 0 ? xp : sp);
        in.h1[i] = *(pos >= 0 ? xp + 1 : sp + (DC - 1));
    }
#pragma unroll
    for (int t = 0; t < kConvTok; ++t)
        in.xs[t] = *reinterpret_cast<const uint32_t*>(p.x + (size_t)(g.t0 + min(tb + min(t, n - 1), g.len - 1)) * L.C + ch);
    // conv_w is [C][dc]: the two channels' 2 dc weights are dc aligned words (ch is even)
    const uint32_t* wp = reinterpret_cast<const uint32_t*>(L.conv_w + (size_t)ch * DC);
#pragma unroll
    for (int i = 0; i < DC; ++i) in.w[i] = wp[i];
}

__device__ __forceinline__ float bf16_half(uint32_t word, int half) {
    return __uint_as_float(half ? (word & 0xffff0000u) : (word << 16));
}

// THRIFTY: sigmoid_r instead of sigmoid_f.
template <int DC, bool SILU, bool THRIFTY = false>
__device__ __forceinline__ void conv_run(ConvIn<DC> in, float (&y0)[kConvTok], float (&y1)[kConvTok]) {
    // Pin the words here: the compiler would otherwise hoist their unpacking up to the loads,
    // which then wait for the data right after issue.
#pragma unroll
    for (int i = 0; i < DC - 1; ++i) { __asm__ volatile("" : "+v"(in.h0[i])); __asm__ volatile("" : "+v"(in.h1[i])); }
#pragma unroll
    for (int t = 0; t < kConvTok; ++t) __asm__ volatile("" : "+v"(in.xs[t]));
#pragma unroll
    for (int i = 0; i < DC; ++i) __asm__ volatile("" : "+v"(in.w[i]));
    float h0[DC - 1], h1[DC - 1], w0[DC], w1[DC];
#pragma unroll
    for (int i = 0; i < DC - 1; ++i) { h0[i] = __uint_as_float(in.h0[i] << 16); h1[i] = __uint_as_float(in.h1[i] << 16); }
#pragma unroll
    for (int i = 0; i < DC; ++i) {
        w0[i] = bf16_half(in.w[i >> 1], i & 1);
        w1[i] = bf16_half(in.w[(DC + i) >> 1], (DC + i) & 1);
    }
#pragma unroll
    for (int t = 0; t < kConvTok; ++t) {
        const float x0 = bf16_half(in.xs[t], 0), x1 = bf16_half(in.xs[t], 1);
        float a0 = 0.0f, a1 = 0.0f;
#pragma unroll
        for (int i = 0; i < DC - 1; ++i) { a0 = fmaf(h0[i], w0[i], a0); a1 = fmaf(h1[i], w1[i], a1); }
        a0 = fmaf(x0, w0[DC - 1], a0);
        a1 = fmaf(x1, w1[DC - 1], a1);
        if constexpr (SILU) {
            a0 = a0 * (THRIFTY ? sigmoid_r(a0) : sigmoid_f(a0));
            a1 = a1 * (THRIFTY ? sigmoid_r(a1) : sigmoid_f(a1));
        }
        y0[t] = a0;
        y1[t] = a1;
#pragma unroll
        for (int i = 0; i < DC - 2; ++i) { h0[i] = h0[i + 1]; h1[i] = h1[i + 1]; }
        h0[DC - 2] = x0;
        h1[DC - 2] = x1;
    }
}

// ---------------------------------------------------------------------------------------
// commit: the rolling conv history of channel ch after sequence s, tokens lo .. lo+len-1
// (len > 0); run by the chain kernel after every read of the old history
// ---------------------------------------------------------------------------------------
// The new history's dc-1 values, loaded (hist_fetch), then stored (hist_put) once they have
// arrived, so that a wave can issue other loads in between.
struct HistNew { uint16_t v[3]; };
__device__ __forceinline__ HistNew hist_fetch(const PrefillParams& p, int ch, int lo, int len, int s) {
    const Layer& L = p.L;
    const uint16_t* st = p.conv_state + ((size_t)s * L.C + ch) * (L.dc - 1);
    // extended history [old (dc-1 values) | the sequence's inputs]; the new history is its
    // last dc-1 entries, i.e. entries len .. len+dc-2. An entry below dc-1 is old history.
    const uint16_t o0 = st[0], o1 = L.dc > 2 ? st[1] : (uint16_t)0, o2 = L.dc > 3 ? st[2] : (uint16_t)0;
    // Entries j >= dc-1 are not stored; their token index is clamped into the sequence, so
    // that no load reaches past its last token.
    HistNew h;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const int ext = len + j;                               // index into the extended history
        const int pos = ext - (L.dc - 1);                      // token position when >= 0
        h.v[j] = pos >= 0 ? p.x[(size_t)(lo + min(pos, len - 1)) * L.C + ch] : (ext == 0 ? o0 : ext == 1 ? o1 : o2);
    }
    return h;
}
__device__ __forceinline__ void hist_put(const PrefillParams& p, int ch, int s, const HistNew& h) {
    const Layer& L = p.L;
    uint16_t* st = p.conv_state + ((size_t)s * L.C + ch) * (L.dc - 1);
    st[0] = h.v[0];
    if (L.dc > 2) st[1] = h.v[1];
    if (L.dc > 3) st[2] = h.v[2];
}

typedef __attribute__((address_space(3))) uint8_t lds_u8;
typedef short v4s __attribute__((ext_vector_type(4)));
// Transposing 8-byte LDS read of 16-bit elements (gfx950 ds_read_b64_tr_b16).
__device__ __forceinline__ uint2 lds_tr16(const lds_u8* a) {
    typedef __attribute__((address_space(3))) v4s lds_v4s;
    return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)a));
}

// 16x16x16 bf16 MFMA operands: A lane l holds A[l%16][4 (l/16) + e], B lane l holds
// B[4 (l/16) + e][l%16], e = 0..3, and the accumulator's lane l holds C[4 (l/16) + r][l%16],
// so an accumulator split to bf16 is the next product's B operand as it stands.
typedef short bf4 __attribute__((ext_vector_type(4)));
struct Split4 { bf4 h, l; };
__device__ __forceinline__ Split4 split4(const v4& x) {
    uint32_t h0, l0, h1, l1;
    split2(x[0], x[1], h0, l0);
    split2(x[2], x[3], h1, l1);
    return Split4{__builtin_bit_cast(bf4, uint2{h0, h1}), __builtin_bit_cast(bf4, uint2{l0, l1})};
}
// c += A B on split operands (hi hi + hi lo + lo hi).
__device__ __forceinline__ v4 mfma16_split(const Split4& a, const Split4& b, v4 c) {
    c = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a.h, b.h, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a.h, b.l, c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a.l, b.h, c, 0, 0, 0);
}
typedef __attribute__((address_space(3))) bf8 lds_bf8;
typedef __attribute__((address_space(3))) v4 lds_v4;

// B operand of one 32-wide k-step from two stacked accumulator tiles (kperm order), split.
__device__ __forceinline__ void split_tiles(const v4& a, const v4& b, bf8& hi, bf8& lo) {
    uint32_t h0, h1, h2, h3, l0, l1, l2, l3;
    split2(a[0], a[1], h0, l0);
    split2(a[2], a[3], h1, l1);
    split2(b[0], b[1], h2, l2);
    split2(b[2], b[3], h3, l3);
    hi = __builtin_bit_cast(bf8, u4x{h0, h1, h2, h3});
    lo = __builtin_bit_cast(bf8, u4x{l0, l1, l2, l3});
}

// Key slots hold each 32-channel block of a key row in kperm order: channels 4 a .. 4 a + 3,
// then 16 + 4 a .. 16 + 4 a + 3, for a = 0..3, i.e. channel 32 b + 16 h + 4 a + e sits at
// position 32 b + 8 a + 4 h + e.
// K fragment (token tile mt, channel k-step ks) of a key slot: A operand of K S. Lane
// (li, lg4) reads row 16 mt + li, channels 32 ks + 4 lg4 .. +3 and 32 ks + 16 + 4 lg4 .. +3:
// the 16 bytes of chunk 4 ks + lg4, stored at chunk (4 ks + lg4) ^ kswz(li) of the row.
__device__ __forceinline__ int k_lane(int li, int lg4, int ks) {
    return li * kPRow + 16 * ((4 * ks + lg4) ^ kswz(li));
}
// kb: the slot plus k_lane(li, lg4, ks).
__device__ __forceinline__ void k_frag(const lds_u8* kb, int mt, bf8& hi, bf8& lo) {
    const int o = mt * 16 * kPRow;
    hi = *(const lds_bf8*)(kb + o);
    lo = *(const lds_bf8*)(kb + kKPlane + o);
}

// K^T fragment (channel tile m, token k-step ks) of a key slot: A operand of K^T Dg, by
// transposing reads (ds_read_b64_tr_b16: within each 16-lane group, lane j receives element
// j & 3 of the 8-byte reads of lanes (j >> 2) + 4 e, e = 0..3). Lane i of lane group g reads
// channels 16 m + 4 (i & 3) .. +3 of token t = 32 ks + 4 g + (i >> 2) (then of the token 16
// later), so it receives channel 16 m + i at tokens 32 ks + 4 g + e (+ 16): entries e (4 + e)
// of its kperm fragment chunk. Those 4 channels are half m & 1 of chunk 4 (m / 2) + (i & 3),
// stored at chunk (4 (m / 2) + (i & 3)) ^ kswz(t) of the row (kswz(t) depends on i and g only).
__device__ __forceinline__ int kt_lane(int i, int g, int mh) {
    const int t = 4 * g + (i >> 2);
    return t * kPRow + 16 * ((4 * mh + (i & 3)) ^ kswz(t));
}
// tb: the slot plus kt_lane(i, g, m / 2); half = m & 1.
__device__ __forceinline__ void kt_frag(const lds_u8* tb, int half, int ks, bf8& hi, bf8& lo) {
    const int o = ks * 32 * kPRow + half * 8;
    const uint2 a = lds_tr16(tb + o), b = lds_tr16(tb + o + 16 * kPRow);
    const uint2 c = lds_tr16(tb + kKPlane + o), d = lds_tr16(tb + kKPlane + o + 16 * kPRow);
    hi = __builtin_bit_cast(bf8, u4x{a.x, a.y, b.x, b.y});
    lo = __builtin_bit_cast(bf8, u4x{c.x, c.y, d.x, d.y});
}


// T' (64 x 64, lower triangular, split) stores its 6 nonzero fragments back to back, (0, 0),
// (1, 0), (2, 0), (2, 1), (3, 0), (3, 1); (0, 0) and (2, 1) pair a diagonal block with a zero
// block, so only entries 0..3 of each lane are stored (8 bytes a lane, 512 a plane). Byte offset
// of a lane's part of one plane:
__host__ __device__ constexpr bool tri_half(int m, int ks) { return (m == 0 && ks == 0) || (m == 2 && ks == 1); }
__device__ __forceinline__ int tri_frag_at(int m, int ks, int plane, int lane) {
    const int off = m == 0 ? 0 : m == 1 ? 1024 : m == 2 ? (ks ? 5120 : 3072) : (ks ? 8192 : 6144);
    return off + (tri_half(m, ks) ? plane * 512 + lane * 8 : plane * 1024 + lane * 16);
}

}  // namespace ixg

// Dequant-fused matmul on the matrix cores for activation rows in the tens to
// thousands (prompt chunks, wide batches) and for MoE segments of such sizes.
//
//   y[M, N] = x16[M, K] . dequant(W[N, K])^T,  fp32 accumulation
//
// Workgroup: W waves (eight at MT = 4, four below), BM = 32 MT activation rows
// by 32 W weight rows (half gate, half up in a GLU launch); a wave owns 32 of
// the weight rows and all BM activation rows.
//  - Weights never pass through LDS: a lane holds its weight row's share of a
//    super-block in registers (half of every 32-value run, 16 contiguous
//    values) and dequantizes straight into the MFMA operand, so every weight
//    is decoded once per workgroup.
//  - Activations do: one super-block (BM rows x 512 bytes) per stage in two
//    LDS buffers, copied by direct-to-LDS loads one stage ahead; every
//    wave reads the same rows, 1 KB per v_mfma_f32_32x32x16_f16.
//  - The B operand is the integer code of kq_mma.h (exact; Q6_K's products
//    above 2048 round to 11 bits there as here); each super-block
//    runs as its own MFMA chain P and folds into the accumulators with the
//    block's fp32 factor.  Q4_K's minimum term multiplies fp32 sub-block sums
//    of the activations, held as three bf16 parts (24 bits), by the integer
//    minimums (exact in bf16) on the matrix cores, and folds with -dmin.
//    The waves share the stage's rows out by sixteen; the sums are used one
//    stage later, behind the stage's only barrier.
//
// Bound by the matrix cores and the decode that shares the SIMDs with them.
// Measured against the small-batch dense kernel and the per-tile gathers: an
// MLP of 2048 bf16 rows (4096 x 12288, Q4_K / Q6_K) 3902 -> 876 us, 706
// TFLOP/s (841 to 881 us over the boxes it ran on); the projections of a layer
// of 333 fp16 rows 830 -> 298 us; an MoE layer of 500 bf16 tokens (128 experts
// of 2048 x 768, 8 a token) 480 -> 294.
//
// Lane l = 32 h + r.  Operand layouts of v_mfma_f32_32x32x16: A row / B column
// r, k values 8 h .. 8 h + 7; result element i: row 8 (i / 4) + 4 h + i % 4,
// column r.  Step (sub, half) of a super-block: lane half h covers values
// 32 sub + 16 h + 8 half .. + 7.
#include <stdlib.h>

#include "kq_gemm.h"
#include "kq_mma.h"

int device_cus();

namespace {

using namespace kqmma;

#define LDSP(T) __attribute__((address_space(3))) T *

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

__device__ __forceinline__ u32x4 lds128(uint32_t a) { return *(const LDSP(u32x4))(uintptr_t)a; }

// 16 bytes a lane from buffer `rs` at voff + soff straight to LDS (lane l's at
// lds + 16 l; the base goes in m0, an operand so that the compiler knows what
// m0 holds).  Written out because the compiler, seeing the builtin, orders
// every LDS read behind it and would drain the copy of the next stage before
// the first fragment of this one; the wait is the explicit one at the stage's
// barrier.  No register receives the load.
__device__ __forceinline__ void dma16(u32x4 rs, uint32_t lds, uint32_t voff, uint32_t soff) {
    asm volatile("s_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :
                 : "{m0}"(lds), "v"(voff), "s"(rs), "s"(soff));
}

// Raw buffer descriptor over `bytes` bytes at `base`, in scalar registers.
__device__ __forceinline__ u32x4 buffer_words(const void *base, uint32_t bytes) {
    const uint64_t p = (uint64_t)base;
    return u32x4{(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)p),
                 (uint32_t)__builtin_amdgcn_readfirstlane((int)((uint32_t)(p >> 32) & 0xFFFFu)),
                 (uint32_t)__builtin_amdgcn_readfirstlane((int)bytes), 0x00020000u};
}

// ---- a lane's share of one super-block of its weight row -------------------
// load(blk, h): the raw bytes.  prep(h): scales, after which a stage replaces
// the block by the next one in place, each register set out again once its
// last step is decoded: early() at any time (into spare registers, the part
// that is decoded last), roll(c) after the steps of sub-blocks 2 c and 2 c + 1
// (c < 3), head() after prep (the scale bytes), commit() at the stage's end.
// frag(sub, half, h): the 8 integer codes of step (sub, half).

template <int CODEC>
struct Share;

template <>
struct Share<KQ_CODEC_Q4_K> {
    u32x4 hdr, q[4], late;
    half2_t sc[4], nb[4];  // scales of sub-blocks 2c, 2c + 1; times -1024 and -64
    uint32_t mlo, mhi;
    float d, dmin;

    __device__ __forceinline__ void load(const uint8_t *blk, int h) {
        hdr = *(const u32x4 *)blk;
#pragma unroll
        for (int c = 0; c < 4; ++c) q[c] = *(const u32x4 *)(blk + 16 + 32 * c + 16 * h);
    }
    __device__ __forceinline__ void early(const uint8_t *blk, int h) { late = *(const u32x4 *)(blk + 16 + 96 + 16 * h); }
    __device__ __forceinline__ void head(const uint8_t *blk) { hdr = *(const u32x4 *)blk; }
    __device__ __forceinline__ void roll(const uint8_t *blk, int h, int c) {
        q[c] = *(const u32x4 *)(blk + 16 + 32 * c + 16 * h);
    }
    __device__ __forceinline__ void commit() { q[3] = late; }
    __device__ __forceinline__ void prep(int) {
        const uint32_t s0 = hdr.y, s1 = hdr.z, s2 = hdr.w;
        const uint32_t scw[2] = {s0 & 0x3F3F3F3Fu, (s2 & 0x0F0F0F0Fu) | ((s0 >> 2) & 0x30303030u)};
        mlo = s1 & 0x3F3F3F3Fu;
        mhi = ((s2 >> 4) & 0x0F0F0F0Fu) | ((s1 >> 2) & 0x30303030u);
        const half2_t k1024 = {(_Float16)1024.f, (_Float16)1024.f};
        const half2_t bias = {(_Float16)-1024.f, (_Float16)-64.f};
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            sc[c] = h2b(kq_bytes_to_h2_biased(scw[c >> 1], (c & 1) ? KQ_SEL_B23 : KQ_SEL_B01)) - k1024;
            nb[c] = sc[c] * bias;
        }
        d = kq_f16_bits_to_f32(hdr.x & 0xFFFFu);
        dmin = kq_f16_bits_to_f32(hdr.x >> 16);
    }
    // The masks and biases of frag's and-ors: the instruction takes one scalar
    // and no literal, so the masks sit in scalar registers and the biases in
    // vector ones.
    struct Consts {
        uint32_t mlow, mhigh, blow, bhigh;
        __device__ __forceinline__ Consts() {
            asm("s_mov_b32 %0, 0x000F000F" : "=s"(mlow));
            asm("s_mov_b32 %0, 0x00F000F0" : "=s"(mhigh));
            asm("v_mov_b32 %0, 0x64006400" : "=v"(blow));
            asm("v_mov_b32 %0, 0x54005400" : "=v"(bhigh));
        }
    };
    // A byte pair in the low bytes of two halves, its low nibbles under 0x64
    // (1024 + q) or its high ones under 0x54 (64 + q): one and-or; then
    // fma(bias + q, sc, -bias sc) = q sc exactly (at most 945).
    __device__ __forceinline__ half8_t frag(int sub, int half, int, const Consts &k, const Iq2Tables &) const {
        const int c = sub >> 1;
        half2_t p[4];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t w = __builtin_amdgcn_perm(0u, q[c][2 * half + i], 0x03010200u);  // bytes 0, 2, 1, 3
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const uint32_t v = j ? w >> 8 : w;
                if (sub & 1)
                    p[2 * i + j] = __builtin_elementwise_fma(h2b((v & k.mhigh) | k.bhigh), bcast(sc[c].y),
                                                             bcast(nb[c].y));
                else
                    p[2 * i + j] = __builtin_elementwise_fma(h2b((v & k.mlow) | k.blow), bcast(sc[c].x),
                                                             bcast(nb[c].x));
            }
        }
        return cat8(p[0], p[1], p[2], p[3]);
    }
    // the eight integer minimums as bf16
    __device__ __forceinline__ u32x4 mins() const {
        u32x4 m;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t w = (i < 2 ? mlo : mhi) >> (16 * (i & 1));
            m[i] = kq_f32x2_to_bf16_bits((float)(w & 0xFFu), (float)((w >> 8) & 0xFFu));
        }
        return m;
    }
    __device__ __forceinline__ float dscale() const { return d; }
};

template <>
struct Share<KQ_CODEC_Q6_K> {
    u32x4 ql[4], qh[2], scw;  // ql[2 n + p]: bytes 64 n + 32 p + 16 h .. + 15
    u32x4 late[3];            // ql[2], ql[3], qh[1] of the next block
    uint32_t dbits;
    half2_t sc[4];  // the lane's scales of sub 2i, 2i + 1
    float d;

    __device__ __forceinline__ static u32x4 at(const uint8_t *p) {
        const u32x4_a2 v = *(const u32x4_a2 *)p;
        return u32x4{v.x, v.y, v.z, v.w};
    }
    __device__ __forceinline__ void load(const uint8_t *blk, int h) {
        roll(blk, h, 1);
        early(blk, h);
        head(blk);
        commit();
    }
    __device__ __forceinline__ void head(const uint8_t *blk) {
        scw = at(blk + 192);
        dbits = (uint32_t)*(const uint16_t *)(blk + 208);
    }
    __device__ __forceinline__ void early(const uint8_t *blk, int h) {
        late[0] = at(blk + 64 + 16 * h);
        late[1] = at(blk + 96 + 16 * h);
        late[2] = at(blk + 160 + 16 * h);
    }
    // sub-blocks 0..3 share their bytes, and so do 4..7
    __device__ __forceinline__ void roll(const uint8_t *blk, int h, int c) {
        if (c != 1) return;
        ql[0] = at(blk + 16 * h);
        ql[1] = at(blk + 32 + 16 * h);
        qh[0] = at(blk + 128 + 16 * h);
    }
    __device__ __forceinline__ void commit() {
        ql[2] = late[0];
        ql[3] = late[1];
        qh[1] = late[2];
    }
    __device__ __forceinline__ void prep(int h) {
        d = kq_f16_bits_to_f32(dbits);
        // scale 2 sub + h: bytes h and 2 + h of word sub / 2
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t w = scw[i] >> (8 * h);
            sc[i] = half2_t{(_Float16)(float)(int8_t)(w & 0xFFu), (_Float16)(float)(int8_t)((w >> 16) & 0xFFu)};
        }
    }
    struct Consts {};
    __device__ __forceinline__ half8_t frag(int sub, int half, int, const Consts &, const Iq2Tables &) const {
        const int n = sub >> 2, qq = sub & 3;
        const half2_t s = bcast((sub & 1) ? sc[sub >> 1].y : sc[sub >> 1].x);
        const half2_t k1056 = {(_Float16)1056.f, (_Float16)1056.f};
        half2_t p[4];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t l = ql[2 * n + (qq & 1)][2 * half + i], hi = qh[n][2 * half + i];
            const uint32_t lo = (qq >= 2 ? l >> 4 : l) & 0x0F0F0F0Fu;
            const uint32_t c = lo | ((2 * qq <= 4 ? hi << (4 - 2 * qq) : hi >> (2 * qq - 4)) & 0x30303030u);
            p[2 * i] = (h2b(kq_bytes_to_h2_biased(c, KQ_SEL_B01)) - k1056) * s;
            p[2 * i + 1] = (h2b(kq_bytes_to_h2_biased(c, KQ_SEL_B23)) - k1056) * s;
        }
        return cat8(p[0], p[1], p[2], p[3]);
    }
    __device__ __forceinline__ float dscale() const { return d; }
};

template <>
struct Share<KQ_CODEC_IQ2_XXS> {
    u32x4 g[4], late;  // groups 2i, 2i + 1: index word, sign | scale word
    uint32_t dbits;
    float d;

    __device__ __forceinline__ static u32x4 at(const uint8_t *p) {
        const u32x4_a2 v = *(const u32x4_a2 *)p;
        return u32x4{v.x, v.y, v.z, v.w};
    }
    __device__ __forceinline__ void load(const uint8_t *blk, int h) {
#pragma unroll
        for (int c = 0; c < 3; ++c) roll(blk, h, c);
        early(blk, h);
        head(blk);
        commit();
    }
    __device__ __forceinline__ void head(const uint8_t *blk) { dbits = (uint32_t)*(const uint16_t *)blk; }
    __device__ __forceinline__ void early(const uint8_t *blk, int) { late = at(blk + 2 + 48); }
    __device__ __forceinline__ void roll(const uint8_t *blk, int, int c) { g[c] = at(blk + 2 + 16 * c); }
    __device__ __forceinline__ void commit() { g[3] = late; }
    __device__ __forceinline__ void prep(int) { d = kq_f16_bits_to_f32(dbits) * 0.125f; }
    struct Consts {};
    __device__ __forceinline__ half8_t frag(int sub, int half, int h, const Consts &, const Iq2Tables &tab) const {
        const uint32_t gw = (sub & 1) ? g[sub >> 1].z : g[sub >> 1].x, aux = (sub & 1) ? g[sub >> 1].w : g[sub >> 1].y;
        const int l = 2 * h + half;
        const u32x4 gm = *(const u32x4 *)tab.grid_h2[(gw >> (8 * l)) & 0xFFu];
        const u32x4 sm = *(const u32x4 *)tab.sign_x2[(aux >> (7 * l)) & 127u];
        const half2_t s = bcast((_Float16)(float)(2u * (aux >> 28) + 1u));
        return cat8(h2b(gm.x ^ sm.x) * s, h2b(gm.y ^ sm.y) * s, h2b(gm.z ^ sm.z) * s, h2b(gm.w ^ sm.w) * s);
    }
    __device__ __forceinline__ float dscale() const { return d; }
};

// ---- the tile ---------------------------------------------------------------

// LDS: two stages of BM rows, two buffers of BM rows' sums (4 parts of 16
// bytes: high, middle, low, zero), the IQ2_XXS tables.
constexpr uint32_t gemm_x_bytes(int MT) { return 32u * MT * 512u; }
constexpr uint32_t gemm_sum_bytes(int MT) { return 32u * MT * 64u; }
constexpr uint32_t gemm_lds_bytes(int MT) {
    return 2 * gemm_x_bytes(MT) + 2 * gemm_sum_bytes(MT) + (uint32_t)sizeof(Iq2Tables);
}

__device__ __forceinline__ floatx16 zero16() {
    floatx16 z;
#pragma unroll
    for (int i = 0; i < 16; ++i) z[i] = 0.f;
    return z;
}

// A lane value the compiler must not carry anything derived from across
// stages: the derived addresses, kept in registers for the whole loop, spilled,
// and a reload waits for every load of the stage.
__device__ __forceinline__ uint32_t per_stage(uint32_t v) {
    asm volatile("" : "+v"(v));
    return v;
}

// Sub-block sums of 16 rows of a stage as bf16 parts, by v_mfma_f32_16x16x32
// with a 0 / 1 selection as A.  Lane group g feeds values of sub-block g (then
// 4 + g), 8 of them a step, so one selection (A row = sub-block) serves four
// steps; element e of lane (g, r) is sub-block 4 g + e of row r (groups 2 and
// 3 hold the zero part).  A step's LDS read is issued ahead of its MFMA.
struct RowSums {
    uint32_t at, out;  // LDS: the lane's first chunk, the row's slot of the sums
    u32x4 v[2];
    floatx4 S;

    int lane;

    __device__ __forceinline__ void start(uint32_t x, uint32_t row0, uint32_t sums) {
        lane = (int)per_stage((uint32_t)kq_lane());
        const int r = lane & 15, g = lane >> 4;
        const uint32_t row = row0 + (uint32_t)r;
        at = x + row * 512u + (((uint32_t)(4 * g) ^ (uint32_t)r) << 4);
        out = sums + row * 64u;
        S = fzero4();
        read(0);
    }
    __device__ __forceinline__ void read(int s) { v[s & 1] = lds128((at ^ (uint32_t)((s & 3) << 4)) + 256u * (s >> 2)); }
    __device__ __forceinline__ void step(int s) {
        const int r = lane & 15, g = lane >> 4;
        S = __builtin_amdgcn_mfma_f32_16x16x32_f16(sum_sel(r, g + (s & 4)), __builtin_bit_cast(half8_t, v[s & 1]), S, 0, 0, 0);
    }
    __device__ __forceinline__ void store() const {
        const int g = lane >> 4;
        const uint32_t key = (uint32_t)(lane & 15) >> 2;
        float hi[4], mid[4], lo[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            hi[e] = (float)(__bf16)S[e];
            mid[e] = (float)(__bf16)(S[e] - hi[e]);
            lo[e] = S[e] - hi[e] - mid[e];
        }
        const u32x2 z = {0u, 0u};
        const u32x2 ph = g < 2 ? u32x2{kq_f32x2_to_bf16_bits(hi[0], hi[1]), kq_f32x2_to_bf16_bits(hi[2], hi[3])} : z;
        const u32x2 pm = {kq_f32x2_to_bf16_bits(mid[0], mid[1]), kq_f32x2_to_bf16_bits(mid[2], mid[3])};
        const u32x2 pl = {kq_f32x2_to_bf16_bits(lo[0], lo[1]), kq_f32x2_to_bf16_bits(lo[2], lo[3])};
        const uint32_t to = out + 8u * (uint32_t)(g & 1);
        *(LDSP(u32x2))(uintptr_t)(to + (((g < 2 ? 0u : 3u) ^ key) << 4)) = ph;
        if (g < 2) {
            *(LDSP(u32x2))(uintptr_t)(to + ((1u ^ key) << 4)) = pm;
            *(LDSP(u32x2))(uintptr_t)(to + ((2u ^ key) << 4)) = pl;
        }
    }
};

// The minimum term of one super-block on 32 rows: acc += nd * (sums . mins),
// with the rows' high and middle parts (lane halves 0, 1) in a[0], low and zero
// in a[1].
__device__ __forceinline__ void add_mins(const u32x4 (&a)[2], const u32x4 &mins, float nd, floatx16 &acc) {
    const bf16x8_t b = __builtin_bit_cast(bf16x8_t, mins);
    floatx16 p = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a[0]), b, zero16(), 0, 0, 0);
    p = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a[1]), b, p, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = __builtin_fmaf(nd, p[i], acc[i]);
}

// Everything of a tile that does not change from stage to stage.
template <int MT, int W, bool GATHER>
struct Tile {
    const uint8_t *w;         // the lane's weight row
    u32x4 xs;                 // buffer over the activation rows
    static constexpr int kCopies = 16 * MT / W;  // 1 KB copies (two rows) of a stage per wave
    // byte offsets of the lane's rows of the wave's copies: rows 2 i + h of a
    // dense tile are xbase + i * xstep; a gathered tile's are its pairs' rows
    uint32_t xbase, xstep;
    uint32_t xrow[GATHER ? kCopies : 1];
    uint32_t rd;              // LDS address of the lane's chunk of step (0, 0) in buffer 0: chunk 4 sub + 2 h + half of
                              // row r is at (chunk ^ r % 16), so step (sub, half)'s is at rd ^ 16 (4 (sub % 4) + half),
                              // 256 bytes on for sub >= 4
    uint32_t sum_rd;          // LDS address of the lane's part h of its row's sums in buffer 0 (^ 32: part 2 + h)
    uint32_t lds;             // the workgroup's LDS
    int wave;
    const Iq2Tables *tab;
};

// Where a lane's part of the stage's copies starts: copy i covers two rows,
// 2 i + h past the wave's first, and chunk l % 32 of LDS holds the row's chunk
// (l % 32) ^ row % 16.
struct CopySource {
    uint32_t row, chunk;

    template <int MT, int W, bool GATHER>
    __device__ __forceinline__ CopySource(const Tile<MT, W, GATHER> &t) {
        const uint32_t l = per_stage((uint32_t)kq_lane());
        row = per_stage(t.xbase);
        chunk = ((l & 31u) ^ (l >> 5) ^ (2u * (uint32_t)(t.wave * t.kCopies) & 15u)) << 4;
    }
};

// The wave's copy i of super-block kb of the activation rows, into buffer `buf`.
template <int MT, int W, bool GATHER>
__device__ __forceinline__ void copy_x(const Tile<MT, W, GATHER> &t, const CopySource &c, int i, int kb, uint32_t buf) {
    const uint32_t dst = (uint32_t)__builtin_amdgcn_readfirstlane(
        (int)(t.lds + buf * gemm_x_bytes(MT) + (uint32_t)(t.wave * t.kCopies + i) * 1024u));
    const uint32_t row = GATHER ? t.xrow[GATHER ? i : 0] : c.row + (uint32_t)i * t.xstep;
    dma16(t.xs, dst, row + (c.chunk ^ (32u * (uint32_t)i & 255u)),
          (uint32_t)__builtin_amdgcn_readfirstlane(kb * 512));
}

__device__ __forceinline__ void stage_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// One super-block: its weights in w, its activations in buffer `buf`; the next
// one's (kb + 1 < kb_end) set out for the other buffer first and for w's
// registers as they fall free.  Sixteen
// MFMA steps with the activation fragments read kAhead steps before their use
// and the weight fragments decoded one step before; Q4_K's sums of this
// stage (steps 0..8) and minimum term of the one before (steps 9 on) ride
// between them.  The barriers keep the scheduler from sinking reads to their
// use or hoisting every fragment of the stage.
template <int CODEC, int MT, int W, bool GATHER>
__device__ __forceinline__ void stage(const Tile<MT, W, GATHER> &t, Share<CODEC> &w, int kb, int kb_end, uint32_t buf,
                                      u32x4 &mins, float &nd, floatx16 (&acc)[MT]) {
    constexpr int kAhead = MT >= 4 ? 1 : 3, kRing = kAhead + 1;
    constexpr int kEvery = Tile<MT, W, GATHER>::kCopies <= 4 ? 2 : 1;  // steps between copies
    constexpr bool kMins = CODEC == KQ_CODEC_Q4_K;
    constexpr bool kMinsLast = MT >= 4;  // once the fragments' registers are free
    constexpr int G = (2 * MT + W - 1) / W;  // 16-row groups of sums per wave
    const int h = kq_lane() >> 5;
    const uint32_t rd = per_stage(t.rd) + buf * gemm_x_bytes(MT);
    const CopySource source(t);
    const uint32_t sums = t.lds + 2 * gemm_x_bytes(MT);
    const uint32_t prev = t.sum_rd + (buf ^ 1u) * gemm_sum_bytes(MT);
    // The last stage reads its own block again, into the buffer and registers
    // nothing reads any more: a load under a branch would make the compiler's
    // waits count for the path without it.
    const int nkb = min(kb + 1, kb_end - 1);
    const int64_t next = (int64_t)nkb * kq_block_bytes(CODEC);
    const typename Share<CODEC>::Consts consts;
    floatx16 P[MT];
    u32x4 a[kRing][MT], ma[2];
    half8_t b[2];
    [[maybe_unused]] RowSums rs[G];
    // step s: pairs of sub-blocks share their bytes, so the order is (pair,
    // half, low / high)
    const auto sub = [](int s) { return 2 * (s >> 2) + (s & 1); };
    const auto half = [](int s) { return (s >> 1) & 1; };
    const auto read_x = [&](int s) {
        const uint32_t at = (rd ^ ((uint32_t)(4 * (sub(s) & 3) + half(s)) << 4)) + 256u * (sub(s) >> 2);
#pragma unroll
        for (int m = 0; m < MT; ++m) a[s % kRing][m] = lds128(at + 16384u * m);
    };
    const auto decode = [&](int s) {
        b[s & 1] = w.frag(sub(s), half(s), h, consts, *t.tab);
    };
    const auto read_mins = [&](int m) {
        ma[0] = lds128(prev + 2048u * m);
        ma[1] = lds128((prev ^ 32u) + 2048u * m);
    };
#pragma unroll
    for (int s = 0; s < kAhead; ++s) read_x(s);
    if constexpr (kMins) {
#pragma unroll
        for (int i = 0; i < G; ++i)
            rs[i].start(t.lds + buf * gemm_x_bytes(MT), 16u * (uint32_t)min(t.wave * G + i, 2 * MT - 1),
                        sums + buf * gemm_sum_bytes(MT));
    }
    w.prep(h);
    decode(0);
#pragma unroll
    for (int s = 0; s < 16; ++s) {
        __builtin_amdgcn_sched_barrier(0);
        if (s + kAhead < 16) read_x(s + kAhead);
        if (s % kEvery == 0 && s / kEvery < t.kCopies) copy_x(t, source, s / kEvery, nkb, buf ^ 1u);
        if (s == 1) w.early(t.w + next, h);
        if (s == 9) w.head(t.w + next);
        if constexpr (kMins) {
#pragma unroll
            for (int i = 0; i < G; ++i) {
                if (s < 7) rs[i].read(s + 1);
                if (s < 8) rs[i].step(s);
                if (s == 9) rs[i].store();  // (a wave past the last group repeats it)
            }
            if (!kMinsLast && s >= 9 && s < 9 + MT) read_mins(s - 9);
        }
        if ((s & 3) == 3 && s < 15) w.roll(t.w + next, h, s >> 2);  // steps up to s are decoded
        if (s < 15) decode(s + 1);
#pragma unroll
        for (int m = 0; m < MT; ++m)
            P[m] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8_t, a[s % kRing][m]), b[s & 1],
                                                          s == 0 ? zero16() : P[m], 0, 0, 0);
        if constexpr (kMins) {
            if (!kMinsLast && s >= 9 && s < 9 + MT) add_mins(ma, mins, nd, acc[s - 9]);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (kMins && kMinsLast) {
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            read_mins(m);
            add_mins(ma, mins, nd, acc[m]);
        }
    }
    if constexpr (kMins) {
        mins = w.mins();
        nd = -w.dmin;
    }
    w.commit();
    const float d = w.dscale();
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[m][i] = __builtin_fmaf(d, P[m][i], acc[m][i]);
    stage_barrier();
}

// acc = the tile over super-blocks [kb0, kb1).
template <int CODEC, int MT, int W, bool GATHER>
__device__ __forceinline__ void accumulate(const Tile<MT, W, GATHER> &t, int kb0, int kb1, floatx16 (&acc)[MT]) {
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[m] = zero16();
    Share<CODEC> w;
    u32x4 mins = {0u, 0u, 0u, 0u};
    float nd = 0.f;
#pragma unroll
    for (int i = 0; i < t.kCopies; ++i) copy_x(t, CopySource(t), i, kb0, 0);
    w.load(t.w + (int64_t)kb0 * kq_block_bytes(CODEC), kq_lane() >> 5);
    if constexpr (CODEC == KQ_CODEC_Q4_K) {
        // the first stage's "stage before" adds nothing: zero sums, zero minimums
        const uint32_t at = t.lds + 2 * gemm_x_bytes(MT) + gemm_sum_bytes(MT);
        for (uint32_t i = threadIdx.x * 16u; i < gemm_sum_bytes(MT); i += 64u * W * 16u)
            *(LDSP(u32x4))(uintptr_t)(at + i) = u32x4{0u, 0u, 0u, 0u};
    }
    stage_barrier();
    int kb = kb0;
    for (;;) {
        stage<CODEC, MT, W, GATHER>(t, w, kb, kb1, 0, mins, nd, acc);
        if (++kb == kb1) break;
        stage<CODEC, MT, W, GATHER>(t, w, kb, kb1, 1, mins, nd, acc);
        if (++kb == kb1) break;
    }
    if constexpr (CODEC == KQ_CODEC_Q4_K) {
        const uint32_t at = t.sum_rd + (uint32_t)((kb1 - kb0 - 1) & 1) * gemm_sum_bytes(MT);
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const u32x4 ma[2] = {lds128(at + 2048u * m), lds128((at ^ 32u) + 2048u * m)};
            add_mins(ma, mins, nd, acc[m]);
        }
    }
}

// ---- epilogues ---------------------------------------------------------------

// GLU tiles: the first half of a workgroup's waves multiply gate columns, the
// second half the same columns of up.  The up waves hand their accumulators
// over through the stage buffers; true for the gate waves, which finish.
template <int MT, int W>
__device__ __forceinline__ bool take_up(uint32_t lds, int wave, floatx16 (&acc)[MT], floatx16 (&up)[MT]) {
    constexpr int H = W / 2;
    const uint32_t at = lds + ((uint32_t)(wave % H) * MT * 4u * 64u + (uint32_t)kq_lane()) * 16u;
    if (wave >= H) {
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                *(LDSP(floatx4))(uintptr_t)(at + (m * 4u + q) * 1024u) =
                    floatx4{acc[m][4 * q], acc[m][4 * q + 1], acc[m][4 * q + 2], acc[m][4 * q + 3]};
    }
    stage_barrier();
    if (wave >= H) return false;
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const floatx4 v = *(const LDSP(floatx4))(uintptr_t)(at + (m * 4u + q) * 1024u);
#pragma unroll
            for (int e = 0; e < 4; ++e) up[m][4 * q + e] = v[e];
        }
    return true;
}

// K slices: every slice of a tile stores its accumulators at the device's
// coherence point and counts its arrival; the last one sums them in slice
// order (bitwise independent of who is last), leaves the counter zero and
// finishes the tile.
template <int MT, int W>
__device__ __forceinline__ bool sum_slices(float *part, uint32_t *counter, int slices, int slice, uint32_t lds,
                                           floatx16 (&acc)[MT]) {
    constexpr int kFloats = MT * 16 * W * 64;  // a tile's accumulators
    float *mine = part + (int64_t)slice * kFloats + threadIdx.x;
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int i = 0; i < 16; ++i)
            __hip_atomic_store(mine + (m * 16 + i) * (W * 64), acc[m][i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    stage_barrier();  // (every store of the workgroup has completed)
    const LDSP(uint32_t) flag = (LDSP(uint32_t))(uintptr_t)lds;
    if (threadIdx.x == 0)
        *(LDSP(uint32_t))(uintptr_t)lds = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    stage_barrier();
    if (*flag != (uint32_t)(slices - 1)) return false;
    floatx16 sum[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) sum[m] = zero16();
    for (int s = 0; s < slices; ++s) {
        const float *p = part + (int64_t)s * kFloats + threadIdx.x;
        floatx16 v[MT];
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int i = 0; i < 16; ++i)
                v[m][i] = __hip_atomic_load(p + (m * 16 + i) * (W * 64), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int i = 0; i < 16; ++i) sum[m][i] += v[m][i];
    }
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[m] = sum[m];
    if (threadIdx.x == 0) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return true;
}

// Row of a tile that result element i of m-tile m holds in this lane.
__device__ __forceinline__ int result_row(int m, int i) { return 32 * m + 8 * (i >> 2) + 4 * (kq_lane() >> 5) + (i & 3); }

template <int MT, int W, bool GATHER>
__device__ __forceinline__ void setup(Tile<MT, W, GATHER> &t, uint8_t *smem, const char *x, uint32_t x_bytes) {
    const int lane = kq_lane(), h = lane >> 5, r = lane & 31;
    t.wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    t.lds = (uint32_t)(uintptr_t)(LDSP(void))smem;
    t.tab = (const Iq2Tables *)(smem + 2 * gemm_x_bytes(MT) + 2 * gemm_sum_bytes(MT));
    t.xs = buffer_words(x, x_bytes);
    t.rd = t.lds + (uint32_t)r * 512u + ((uint32_t)((2 * h) ^ (r & 15)) << 4);
    // a row's four parts of sums swap places by row, so that sixteen rows spread over the banks
    t.sum_rd = t.lds + 2 * gemm_x_bytes(MT) + (uint32_t)r * 64u + ((uint32_t)(h ^ ((r >> 2) & 3)) << 4);
}

template <int MT, int W, bool GATHER>
__device__ __forceinline__ void accumulate_codec(const Tile<MT, W, GATHER> &t, int codec, int kb0, int kb1,
                                                 floatx16 (&acc)[MT]) {
    switch (codec) {
    case KQ_CODEC_Q4_K: accumulate<KQ_CODEC_Q4_K, MT, W, GATHER>(t, kb0, kb1, acc); break;
    case KQ_CODEC_Q6_K: accumulate<KQ_CODEC_Q6_K, MT, W, GATHER>(t, kb0, kb1, acc); break;
    default:
        load_iq2_tables(*(Iq2Tables *)t.tab);
        accumulate<KQ_CODEC_IQ2_XXS, MT, W, GATHER>(t, kb0, kb1, acc);
        break;
    }
}

// Workgroups go to the eight XCDs in turn: XCD b % 8 takes a contiguous range
// of the tiles, so that neighbours share its L2.  -1: none left.
__device__ __forceinline__ int xcd_tile(int tiles) {
    const int per = (tiles + 7) / 8, i = (int)blockIdx.x >> 3;
    const int tile = ((int)blockIdx.x & 7) * per + i;
    return i < per && tile < tiles ? tile : -1;
}

// ---- dense ------------------------------------------------------------------

struct GemmProblem {
    const uint8_t *w, *w1;  // w1: the up matrix of a GLU launch
    const char *x;
    const int32_t *x_exp;
    void *y;
    int64_t w_row_bytes, y_stride;
    uint32_t x_row_bytes, x_bytes;
    int32_t M, N, K, codec;
    int32_t m_tiles, begin;  // row tiles; first tile of this problem
};

struct GemmArgs {
    GemmProblem p[KQ_MAX_GROUP];
    int32_t n_problems, tiles, y_dtype, act, slices;
    float *part;         // [tiles][slices] partial tiles
    uint32_t *counters;  // one per tile
};

template <int MT, int W, bool GLU>
__global__ __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(2))) void kq_gemm_kernel(GemmArgs a) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    constexpr int BM = 32 * MT, BN = 32 * (GLU ? W / 2 : W);
    const int unit = xcd_tile(a.tiles * a.slices);
    if (unit < 0) return;  // uniform over the workgroup
    const int tile = unit / a.slices, slice = unit - tile * a.slices;
    GemmProblem p = a.p[0];
#pragma unroll
    for (int i = 1; i < KQ_MAX_GROUP; ++i)
        if (i < a.n_problems && tile >= a.p[i].begin) p = a.p[i];
    const int local = tile - p.begin;
    const int nt = local / p.m_tiles, mt = local - nt * p.m_tiles;  // row tiles first: one weight panel for all of them
    Tile<MT, W, false> t;
    setup(t, smem, p.x, p.x_bytes);
    const int lane = kq_lane(), h = lane >> 5, r = lane & 31;
    const int m0 = mt * BM, col = nt * BN + (GLU ? t.wave % (W / 2) : t.wave) * 32 + r;
    // rows past M lie past the buffer: they read as zeros and touch no memory
    t.xbase = (uint32_t)(m0 + 2 * t.wave * t.kCopies + h) * p.x_row_bytes;
    t.xstep = 2u * p.x_row_bytes;
    t.w = (GLU && t.wave >= W / 2 ? p.w1 : p.w) + (int64_t)min(col, p.N - 1) * p.w_row_bytes;
    const int nb = p.K / KQ_QK;
    floatx16 acc[MT];
    accumulate_codec(t, p.codec, slice * nb / a.slices, (slice + 1) * nb / a.slices, acc);
    [[maybe_unused]] floatx16 up[MT];
    if constexpr (GLU) {
        if (!take_up<MT, W>(t.lds, t.wave, acc, up)) return;
    } else if (a.slices > 1) {
        if (!sum_slices<MT, W>(a.part + (int64_t)tile * a.slices * (MT * 16 * W * 64), a.counters + tile, a.slices, slice,
                               t.lds, acc))
            return;
    }
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int row = m0 + result_row(m, i);
            if (row >= p.M || col >= p.N) continue;
            const int e = p.x_exp ? p.x_exp[row] : 0;
            float v = ldexpf(acc[m][i], e);
            if constexpr (GLU) v = kq_glu(a.act, v, ldexpf(up[m][i], e), 0.f, 0.f, 0.f, 0.f);
            kq_store_out(p.y, a.y_dtype, (int64_t)row * p.y_stride + col, v);
        }
}

// ---- MoE segments -------------------------------------------------------------

// A tile is up to BM rows of one expert's segment by BN of its weight rows.
// Tiles run chunk of rows first, column tile within: the chunk table (chunks
// before each segment) is a wave scan over the segments, each wave for itself.
template <int MT, int W, bool GLU>
__global__ __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(2))) void kq_gemm_gather_kernel(KqGemmGather a) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    constexpr int BM = 32 * MT, BN = 32 * (GLU ? W / 2 : W);
    const int lane = kq_lane(), h = lane >> 5, r = lane & 31;
    const int n_tiles = (a.N + BN - 1) / BN;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    // pairs whose expert id is out of range (never routed) get zeros
    if ((int)blockIdx.x < n_tiles) {
        const int per = BN / W;  // columns per wave
        const int c = (int)blockIdx.x * BN + wave * per + lane;
        kq_for_unrouted(a.pair_order + a.n_pairs, a.n_pairs, [&](int p) {
            if (lane < per && c < a.N)
                kq_store_out(a.y, a.y_dtype, (int64_t)(p + (a.y_skip ? p / a.y_skip : 0)) * a.y_stride + c, 0.f);
        });
    }
    const int S = a.seg_info[0];
    const int32_t *start = a.seg_info + 1 + a.n_experts;
    int chunks = 0;
    for (int s0 = 0; s0 < S; s0 += 64) {
        const int s = s0 + lane;
        int n = s < S ? (start[s + 1] - start[s] + BM - 1) / BM : 0;
        for (int off = 32; off > 0; off >>= 1) n += __shfl_xor(n, off);
        chunks += n;
    }
    const int tile = xcd_tile(__builtin_amdgcn_readfirstlane(chunks) * n_tiles);
    if (tile < 0) return;  // uniform over the workgroup
    const int chunk = tile / n_tiles, nt = tile - chunk * n_tiles;
    int seg = 0, first = 0;  // the chunk's segment, its first row
    for (int s0 = 0, base = 0; s0 < S; s0 += 64) {
        const int s = s0 + lane;
        const int n = s < S ? (start[s + 1] - start[s] + BM - 1) / BM : 0;
        int inc = n;
        for (int off = 1; off < 64; off <<= 1) {
            const int v = __shfl_up(inc, off);
            if (lane >= off) inc += v;
        }
        const uint64_t hit = __ballot(chunk >= base + inc - n && chunk < base + inc);
        if (hit) {
            const int src = __builtin_ctzll(hit);
            seg = s0 + src;
            first = (chunk - base - __shfl(inc - n, src)) * BM;
            break;
        }
        base += __shfl(inc, 63);
    }
    seg = __builtin_amdgcn_readfirstlane(seg);
    first = __builtin_amdgcn_readfirstlane(first);
    const int expert = a.seg_info[1 + seg];
    const int begin = start[seg] + first, rows = min(start[seg + 1] - begin, BM);
    Tile<MT, W, true> t;
    setup(t, smem, a.x, a.x_bytes);
#pragma unroll
    for (int i = 0; i < t.kCopies; ++i) {
        const int row = 2 * (t.wave * t.kCopies + i) + h;
        const int pair = a.pair_order[begin + min(row, rows - 1)];
        const uint32_t xr = (uint32_t)(pair / a.x_pair_div + (a.x_skip ? pair / a.x_skip : 0));
        t.xrow[i] = row < rows ? xr * a.x_row_bytes : 0x80000000u;  // past the buffer: zeros, no memory touched
    }
    t.xbase = t.xstep = 0;
    const int col = nt * BN + (GLU ? t.wave % (W / 2) : t.wave) * 32 + r;
    t.w = (GLU && t.wave >= W / 2 ? a.w1 : a.w0) + (int64_t)expert * a.w_expert_bytes +
          (int64_t)min(col, a.N - 1) * a.w_row_bytes;
    floatx16 acc[MT];
    accumulate_codec(t, a.codec, 0, a.K / KQ_QK, acc);
    [[maybe_unused]] floatx16 up[MT];
    if constexpr (GLU) {
        if (!take_up<MT, W>(t.lds, t.wave, acc, up)) return;
    }
    const int64_t bo = (int64_t)expert * a.b_stride + min(col, a.N - 1);
    const float b0 = a.b0 ? a.b0[bo] : 0.f, b1 = a.b1 ? a.b1[bo] : 0.f;
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int row = result_row(m, i);
            if (row >= rows || col >= a.N) continue;
            const int pair = a.pair_order[begin + row];
            const int e = a.x_exp ? a.x_exp[pair / a.x_pair_div + (a.x_skip ? pair / a.x_skip : 0)] : 0;
            float v = ldexpf(acc[m][i], e);
            if constexpr (GLU)
                v = kq_glu(a.act, v, ldexpf(up[m][i], e), a.limit, a.alpha, b0, b1);
            else
                v += b0;
            kq_store_out(a.y, a.y_dtype, (int64_t)(pair + (a.y_skip ? pair / a.y_skip : 0)) * a.y_stride + col, v);
        }
}

// ---- host ---------------------------------------------------------------------

int env_int(const char *name, int dflt) {
    const char *s = getenv(name);
    return (s && *s) ? atoi(s) : dflt;
}

int set_lds(const void *fn, int MT) {
    return hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)gemm_lds_bytes(MT)) == hipSuccess
               ? KQ_OK
               : KQ_ERR_LAUNCH_FAILED;
}

template <int MT, int W, bool GLU>
int launch(const GemmArgs &a, hipStream_t s) {
    if (const int rc = set_lds((const void *)kq_gemm_kernel<MT, W, GLU>, MT)) return rc;
    hipLaunchKernelGGL((kq_gemm_kernel<MT, W, GLU>), dim3(8 * ((a.tiles * a.slices + 7) / 8)), dim3(64 * W),
                       gemm_lds_bytes(MT), s, a);
    return hipGetLastError() == hipSuccess ? KQ_OK : KQ_ERR_LAUNCH_FAILED;
}

template <bool GLU>
int launch_mt(int mt, const GemmArgs &a, hipStream_t s) {
    return mt == 4 ? launch<4, 8, GLU>(a, s) : mt == 2 ? launch<2, 4, GLU>(a, s) : launch<1, 4, GLU>(a, s);
}

template <int MT, int W, bool GLU>
int launch_gather(const KqGemmGather &a, int grid, hipStream_t s) {
    if (const int rc = set_lds((const void *)kq_gemm_gather_kernel<MT, W, GLU>, MT)) return rc;
    hipLaunchKernelGGL((kq_gemm_gather_kernel<MT, W, GLU>), dim3(grid), dim3(64 * W), gemm_lds_bytes(MT), s, a);
    return hipGetLastError() == hipSuccess ? KQ_OK : KQ_ERR_LAUNCH_FAILED;
}

int tile_cols(int mt, bool glu) { return (mt == 4 ? 256 : 128) / (glu ? 2 : 1); }

// Workgroups a launch may have: its threads are counted in 32 bits, and the
// grid is rounded up to the eight XCDs.
int64_t max_groups(int mt) { return (((int64_t)1 << 32) - 1) / (mt == 4 ? 512 : 256) - 8; }

// Tile height and K slices of a dense launch.
struct Plan {
    int mt, slices, tiles;
    int64_t part_bytes;  // of all tiles' slices
};

// Microseconds per super-block of a launch whose tiles come to `w` per CU
// (w >= 1: the fuller of the last round's two halves).  Measured on Q4_K (Q6_K
// in brackets) at K = 4096 / 12288: the 128 x 256 tile holds a CU alone, 4.0
// for one and 5.6 for each further; two 64 x 128 tiles share a CU, 1.95 for
// one, 3.5 (4.1) for two; three 32 x 128 tiles do, 1.6 for one, 3.5 (5.0) for
// three.
double stage_us(int mt, int codec, double tiles, int cus) {
    double w = tiles / cus;
    if (w < 1) w = 1;
    const double c = (double)(int64_t)(w + 0.999999), half = 0.5 * (w + c);
    const bool q6 = codec == KQ_CODEC_Q6_K;
    if (mt == 4) return 4.0 + 5.6 * (c - 1);
    if (mt == 2) return 0.3 + 1.65 * (q6 ? 1.18 : 1.0) * half;
    return 0.45 + 1.15 * (q6 ? 1.45 : 1.0) * half;
}

// The plan that the figures above make the shortest.  K slices (of at least
// four super-blocks) only without a GLU, in the counters' range, and with their
// partial tiles written and read once each at ~3 TB/s behind ~4 us of stores,
// arrivals and loads.
Plan make_plan(const kq_matmul_problem *ps, int n, bool glu) {
    const int cus = device_cus(), forced = env_int("GMLX_KQ_GEMM_MT", 0), forced_s = env_int("GMLX_KQ_GEMM_S", 0);
    Plan best{0, 1, 0, 0};
    double best_us = 0;
    for (int mt = 4; mt >= 1; mt /= 2) {
        if (forced && mt != forced) continue;
        int64_t tiles = 0;
        int nb_min = 1 << 30, nb_max = 0, codec = KQ_CODEC_Q4_K;
        for (int i = 0; i < n; ++i) {
            tiles += (int64_t)((ps[i].M + 32 * mt - 1) / (32 * mt)) *
                     ((ps[i].N + tile_cols(mt, glu) - 1) / tile_cols(mt, glu));
            const int nb = ps[i].K / KQ_QK;
            nb_min = nb < nb_min ? nb : nb_min;
            nb_max = nb > nb_max ? nb : nb_max;
            if (ps[i].codec == KQ_CODEC_Q6_K) codec = KQ_CODEC_Q6_K;
        }
        for (int s = 1; s <= 8; ++s) {
            if (forced_s && s != forced_s && !glu) continue;
            if (s > 1 && (glu || nb_min < 4 * s || tiles > (int64_t)(KQ_MATMUL_COUNTER_BYTES / 4))) break;
            if (tiles * s > max_groups(mt)) break;
            const int64_t part = s > 1 ? tiles * s * (mt * 16 * (mt == 4 ? 8 : 4) * 64 * 4) : 0;
            const double us = ((double)nb_max / s + 1.5) * stage_us(mt, codec, (double)tiles * s, cus) +
                              (s > 1 ? 4.0 + 2e-6 * (double)part / 3.0 : 0.0);
            if (!best.mt || us < best_us) {
                best = Plan{mt, s, (int)tiles, part};
                best_us = us;
            }
        }
    }
    return best;
}

void set_problem(GemmProblem &p, const kq_matmul_problem &q, const int32_t *x_exp, int mt, bool glu, int &tiles) {
    p.w = (const uint8_t *)q.w;
    p.w1 = nullptr;
    p.x = (const char *)q.x;
    p.x_exp = x_exp;
    p.y = q.y;
    p.w_row_bytes = q.w_row_bytes;
    p.y_stride = q.y_row_stride;
    p.x_row_bytes = (uint32_t)q.x_row_stride * 2;
    p.x_bytes = (uint32_t)(((int64_t)(q.M - 1) * q.x_row_stride + q.K) * 2);
    p.M = q.M;
    p.N = q.N;
    p.K = q.K;
    p.codec = q.codec;
    p.m_tiles = (p.M + 32 * mt - 1) / (32 * mt);
    p.begin = tiles;
    tiles += p.m_tiles * ((p.N + tile_cols(mt, glu) - 1) / tile_cols(mt, glu));
}

// 32-bit activation offsets, with room for the rows of a tile past M
bool addressable(int64_t rows, int64_t row_stride) { return rows * row_stride * 2 < (int64_t)1 << 31; }

}  // namespace

// Small launches of short rows stay on the dense kernel: fewer than 8
// super-blocks take no K slices, so a launch is one tile's walk over K long,
// and a Q6_K step takes 1.6 us here against 1.3 there, as long as that
// kernel's workgroups (32 columns by 64 rows) fit one a CU.  Theirs / these,
// 65 to 128 rows (us): Q6_K, 1024 rows of 256 values 8.7 / 8.9, of 1024 12.6 /
// 13.8, of 1792 17.1 / 22.1, of 2048 (two slices) 18.1 / 16.2; 4096 rows of
// 1024 13.0 / 14.5, and 18.6 / 14.6 at 129 rows, where they no longer fit; a
// q|k|v group (Q4_K, V in Q6_K) of 4096 rows of 1024 13.0 / 14.5; IQ2_XXS, 512
// rows of 1536 13.6 / 14.8, of 1024 11.7 / 11.8.  Everywhere else past 64 rows
// the tiles are level or ahead: 65 rows by 4096 x 4096 28.8 / 20.2 in Q4_K,
// 28.6 / 24.1 in Q6_K, 25.1 / 20.4 in IQ2_XXS; 12288 x 4096 68 / 33, 74 / 49,
// 58 / 33; Q4_K by 1024 x 1024 12.2 / 10.1.
static bool dense_kernel_pays(const kq_matmul_problem *ps, int n) {
    bool slow = false;
    int64_t workgroups = 0;
    for (int i = 0; i < n; ++i) {
        const int nb = ps[i].K / KQ_QK;
        if (nb >= 8) return false;
        slow = slow || ps[i].codec == KQ_CODEC_Q6_K || (ps[i].codec == KQ_CODEC_IQ2_XXS && nb > 4);
        workgroups += (int64_t)((ps[i].N + 31) / 32) * ((ps[i].M + 63) / 64);
    }
    return slow && workgroups <= device_cus();
}

bool kq_gemm_eligible(const kq_matmul_problem *ps, int n) {
    for (int i = 0; i < n; ++i)
        if (ps[i].M <= 64 || !addressable(ps[i].M, ps[i].x_row_stride)) return false;
    const int mode = env_int("GMLX_KQ_GEMM", 1);
    if (n <= 0 || mode == 0) return false;
    if (mode != 2 && !env_int("GMLX_KQ_GEMM_MT", 0) && dense_kernel_pays(ps, n)) return false;
    return make_plan(ps, n, false).mt != 0;
}

size_t kq_gemm_part_bytes(const kq_matmul_problem *ps, int n) {
    return kq_gemm_eligible(ps, n) ? (size_t)make_plan(ps, n, false).part_bytes : 0;
}

int kq_gemm_launch(const kq_matmul_problem *ps, const int32_t *const *exps, int n, int y_dtype, uint32_t *counters,
                   float *part, hipStream_t s) {
    Plan plan = make_plan(ps, n, false);
    if (!part) plan.slices = 1;
    GemmArgs a;
    int tiles = 0;
    for (int i = 0; i < n; ++i) set_problem(a.p[i], ps[i], exps[i], plan.mt, false, tiles);
    a.n_problems = n;
    a.tiles = tiles;
    a.y_dtype = y_dtype;
    a.act = 0;
    a.slices = plan.slices;
    a.part = part;
    a.counters = counters;
    return launch_mt<false>(plan.mt, a, s);
}

bool kq_gemm_glu_eligible(const kq_matmul_problem &gate) {
    return gate.M > 64 && addressable(gate.M, gate.x_row_stride) && env_int("GMLX_KQ_GEMM", 1) != 0 &&
           make_plan(&gate, 1, true).mt != 0;
}

int kq_gemm_glu_launch(const kq_matmul_problem &gate, const void *w_up, const int32_t *x_exp, int act, int y_dtype,
                       hipStream_t s) {
    const Plan plan = make_plan(&gate, 1, true);
    GemmArgs a;
    int tiles = 0;
    set_problem(a.p[0], gate, x_exp, plan.mt, true, tiles);
    a.p[0].w1 = (const uint8_t *)w_up;
    a.n_problems = 1;
    a.tiles = tiles;
    a.y_dtype = y_dtype;
    a.act = act;
    a.slices = 1;
    a.part = nullptr;
    a.counters = nullptr;
    return launch_mt<true>(plan.mt, a, s);
}

// Rows per tile of a gather from the mean segment: 32 up to 28 (a layer at
// 18.8 rows per expert: 198 us against 232 with 64-row tiles), 64 past it (at
// 32 rows over 8 experts 195 us against 246; over 128 experts the two are
// level, 263 against 258).
static int gather_mt(int64_t n_pairs, int slots) {
    const int forced = env_int("GMLX_KQ_GEMM_MT", 0);
    return forced ? (forced == 1 ? 1 : 2) : n_pairs > 28 * (int64_t)slots ? 2 : 1;
}

// Whether a gather is shorter on these tiles than on the kernel it would take
// otherwise (`streams`: the streaming gather, else the per-tile ones).
//
// Those read a segment's weights in less time but multiply 8 or 16 rows at a
// time.  Launches of more tiles than CUs, whole layers (us, theirs / these):
// 128 experts of 2048 x 768, 156 / 169 at 6.2 pairs per expert, 170 / 173 at
// 8, 230 / 181 at 12.5, 457 / 258 at 31; 256 IQ2_XXS experts of 7168 x 2048,
// 1250 / 1632 at 4, 1726 / 1688 at 8, 3332 / 1912 at 16; 16 IQ2_XXS experts
// of 4096 x 1024, 45 / 51 at 8.5, 55 / 52 at 12.  So the line is 8 pairs per
// expert, 10 for IQ2_XXS.
//
// A launch of at most one tile a CU (few experts or narrow ones, above all the
// shared expert, one segment of all the tokens) is one tile's walk over K
// long, while the other kernels cut N by sixteens and long K over four waves:
// there both times are estimated, and the tiles have to win by 8 %.  Fitted to
// 374 launches (1 to 16 experts, 8.5 to 1024 rows each, N 512 to 8192, K 512
// to 8192, the three codecs) and tried on 160 more: 188 of the 374 ran over
// 3 % slower on these tiles, by up to 4.2 times; with the rule 4 of all 534 do,
// by 4 to 15 %.  Theirs / these, one expert's
// GLU of 768 x 2048 in Q4_K: 9.1 / 19.0 at 24 rows, 22 / 29 at 256, 36 / 30 at
// 512; 2048 x 7168: 23 / 41, 152 / 62 and 299 / 71; its down projection in
// Q6_K: 24 / 26, 146 / 36 and 287 / 51.
static bool gather_pays(const KqGemmGather &a, bool streams) {
    const bool q6 = a.codec == KQ_CODEC_Q6_K, iq2 = a.codec == KQ_CODEC_IQ2_XXS, glu = a.w1 != nullptr;
    if (a.n_pairs <= (iq2 ? 10 : 8) * (int64_t)a.n_experts) return false;
    const int cus = device_cus(), slots = a.n_experts < a.n_pairs ? a.n_experts : a.n_pairs;
    const double mean = (double)a.n_pairs / slots;
    const int mt = gather_mt(a.n_pairs, slots);
    const int64_t n_tiles = (a.N + tile_cols(mt, glu) - 1) / tile_cols(mt, glu);
    if (slots * (1 + (int64_t)((a.n_pairs - 1) / ((int64_t)slots * 32 * mt))) * n_tiles > cus) return true;
    const double nb = a.K / KQ_QK;
    const double tiles = mt == 1 ? 10 + nb * (q6 ? 2.05 : iq2 ? 1.4 : 1.1) : 13 + nb * (q6 ? 2.5 : iq2 ? 1.75 : 1.6);
    double theirs;
    if (streams) {
        // by the weights read and the rows multiplied, per 2 x 768 x 2048 weights of an expert
        theirs = 8 + 2.0 * a.N * a.K / (2.0 * 768 * 2048) * (0.35 * slots + 0.07 * a.n_pairs);
    } else {
        // a unit's chunks of 16 rows (segments scatter about the mean) by its
        // steps through K, times the rounds of units
        const int chunks = slots == 1 ? (a.n_pairs + 15) / 16 : (int)(mean / 16) + 1;
        const double waves = (double)slots * ((a.N + 15) / 16) * (nb > 8 ? 4 : 1) * (glu ? 1.5 : 1.0) *
                             (iq2 ? 0.8 : 1.0) / (4.0 * cus);
        theirs = 7 + 1.2 * chunks * (nb > 8 ? nb / 4 : nb) * (waves > 1 ? waves : 1);
    }
    return theirs > 1.08 * tiles;
}

// Workgroups of a gather: they bound every chunk of every segment.
static int64_t gather_groups(const KqGemmGather &a, int mt) {
    const int slots = a.n_experts < a.n_pairs ? a.n_experts : a.n_pairs, cols = tile_cols(mt, a.w1 != nullptr);
    return ((int64_t)a.n_pairs / (32 * mt) + slots) * ((a.N + cols - 1) / cols);
}

bool kq_gemm_gather_eligible(const KqGemmGather &a, int64_t x_rows, int64_t x_row_stride, bool streams) {
    const int mode = env_int("GMLX_KQ_GEMM", 1);
    const int mt = gather_mt(a.n_pairs, a.n_experts < a.n_pairs ? a.n_experts : a.n_pairs);
    return mode != 0 && addressable(x_rows, x_row_stride) && gather_groups(a, mt) <= max_groups(mt) &&
           (mode == 2 || gather_pays(a, streams));
}

int kq_gemm_gather_launch(const KqGemmGather &a, hipStream_t s) {
    const bool glu = a.w1 != nullptr;
    const int mt = gather_mt(a.n_pairs, a.n_experts < a.n_pairs ? a.n_experts : a.n_pairs);
    const int grid = 8 * (int)((gather_groups(a, mt) + 7) / 8);
    if (mt == 2) return glu ? launch_gather<2, 4, true>(a, grid, s) : launch_gather<2, 4, false>(a, grid, s);
    return glu ? launch_gather<1, 4, true>(a, grid, s) : launch_gather<1, 4, false>(a, grid, s);
}

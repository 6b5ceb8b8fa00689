// GGUF (Q8_0, IQ3_S) products y_j = W x_j for 1..8 inputs on the matrix cores (matvec_cols_*).
//
// Both formats' weights are a scale times small integers (Q8_0: codes of 8 bits, a scale a 32-block; IQ3_S: grid value * sign *
// (1 + 2 s), at most 465, one scale a 256-block), which f16 holds exactly.  A row of W is a column of operand B of
// v_mfma_f32_16x16x32_f16: lane 16 g + r holds 8 weights of row r.  The inputs ride on the rows of operand A in three f16
// parts of 11 bits, scaled by the power of two that takes the largest magnitude of their 256 columns to [2^14, 2^15), and the
// second and third part 2^11 and 2^22 times more, so that they do not run under f16's smallest value: together they are the
// f32 exactly down to 2^-37 of the largest, and within 2^-61 of the largest below.  An IQ3_S block's weights are between 1 and
// 465 times its scale, so that is far under the rounding of the f32 sums which the largest input is part of; a Q8_0 code may be
// zero where the largest input meets it, so what the parts leave is multiplied on the vector unit (gg_rest): no size of one
// input costs another a bit, as with f32 multiply-adds.  Token t's parts are rows 4 t .. 4 t + 2, so its three sums come out in
// one lane (16 t + r), where two multiply-adds and the block's scale, one more, put them together.  Products are exact and
// sums are f32; an integer is decoded once for up to 8 inputs (1.3 vector instructions a Q8_0 weight, 4 an IQ3_S one, where
// the vector unit alone takes 2 and 8 and one more a token).
//
// A wave takes 256-column chunks and keeps a chunk's input parts in registers while it goes over the workgroup's tiles of 16
// rows: the parts are made once a chunk, not once a chunk and row group, and a matrix of few rows still spreads over all its
// chunks.  A Q8_0 tile's chunk comes in 16-byte loads along the rows and is turned round in a strip of LDS of the wave's own
// (loads of a lane's own 8 codes, 16 rows apart, stopped at 2.2 TB/s without any product).
// Measured: Q8_0, 8201 rows of 3072 columns, 5 inputs: 10.9 us a call (2.5 TB/s; 25 with the parts made for every 32 rows and
// loads of a lane's own codes, 41 on the vector unit).  What is left is the chain of a workgroup's start, an input's parts and two
// or three tiles, not the memory: a CU runs one such workgroup at a time.  So the parts take few instructions: the largest
// magnitude by whole-number DPP steps into a scalar, then five mixed-precision multiply-adds an input (2048 x 8192, 3 inputs: 11.4
// -> 10.7 us), and their rest for free.  Tiles of 8 or 4 rows for matrices of few rows measured the same as 16.
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef u32 u32x2b __attribute__((ext_vector_type(2), aligned(2)));   // GGUF rows are only 2-byte aligned
typedef u32 u32x4b __attribute__((ext_vector_type(4), aligned(2)));

#define GG_PITCH 264                 /* f16 from one A row of the parts to the next: 256 and a shift of four banks */
#define GG_STRIP (12 * GG_PITCH / 2) /* words of a wave's strip: four inputs' parts, then the weights */

__device__ __forceinline__ f16x2 gg_pair(u32 v) { return __builtin_bit_cast(f16x2, v); }
__device__ __forceinline__ u32 gg_bits(f16x2 v) { return __builtin_bit_cast(u32, v); }

// The three parts' sums put together, in units of the first one's.
__device__ __forceinline__ float gg_sum(const f32x4& s) { return __builtin_fmaf(__builtin_fmaf(s[2], 0x1p-11f, s[1]), 0x1p-11f, s[0]); }

// What a wave's LDS stores and loads of its own strip need between them: the compiler keeps their order, the chip does anyway.
__device__ __forceinline__ void gg_order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// 16 rows x 256 columns of a wave: load() requests them, stage() makes them readable, products() adds
// sum of the chunk for token 4 G + lane / 16 and row lane % 16 to out[G], in units of the inputs' scale.
struct GgQ8 {
    static constexpr u32 QK = 32, BB = 34, CHUNK = 272;   // bytes of a 256-column chunk: 17 pieces of 16
    static constexpr u32 PITCH = 72;                      // words of a row in the strip: 68 and a shift of four banks
    static constexpr bool grid = false, zeros = true;     // a table to look weights up in; weights that may be zero
    static constexpr u32 part_at(u32 q, u32 g) { return 32 * q + 8 * g; }   // first column of the lane's 8 in instruction q
    u32x4b v[5];
    u32 at[2];   // the pieces' rows and places in their rows, five bits each, three pieces a word
    __device__ __forceinline__ void init(u32 lane) {
        at[0] = at[1] = 0;
#pragma unroll
        for (u32 i = 0; i < 5; i++) {
            const u32 p = lane + 64 * i;
            at[i / 3] |= (p % 17 + p / 17 * 32) << (10 * (i % 3));
        }
    }
    __device__ __forceinline__ u32 place(int i) const { return __builtin_amdgcn_ubfe(at[i / 3], 10 * (i % 3), 5); }
    __device__ __forceinline__ u32 row(int i) const { return __builtin_amdgcn_ubfe(at[i / 3], 10 * (i % 3) + 5, 5); }
    __device__ __forceinline__ void load(const u8* __restrict__ w, u32 rb, u32 first, u32 rows, u32 col, u32 lane) {
        if (rb < CHUNK) return;
        const u8* base = w + (u64) first * rb + col / 32 * 34;
        const u32 rmost = rows - 1 - first;
#pragma unroll
        for (int i = 0; i < 2; i++) asm volatile("" : "+v"(at[i]));   // the addresses are a few operations: not kept
#pragma unroll
        for (int i = 0; i < 5; i++)
            if (i < 4 || lane < 16) v[i] = *(const u32x4b*) (base + (u64) min(row(i), rmost) * rb + place(i) * 16);
    }
    __device__ __forceinline__ void stage(u32* strip, const u8* __restrict__ w, u32 rb, u32 first, u32 rows, u32 lane) const {
        if (rb < CHUNK) {
            // rows shorter than a chunk: halfword by halfword, zeros (codes and scales) after a row's end
#pragma unroll 1
            for (u32 i = lane; i < 16 * (CHUNK / 2); i += 64) {
                const u32 r = i / (CHUNK / 2), h = i % (CHUNK / 2);
                ((u16*) strip)[r * 2 * PITCH + h] = 2 * h < rb ? *(const u16*) (w + (u64) min(first + r, rows - 1) * rb + 2 * h) : (u16) 0;
            }
        } else {
#pragma unroll
            for (int i = 0; i < 5; i++)
                if (i < 4 || lane < 16) *(u32x4*) (strip + row(i) * PITCH + place(i) * 4) = u32x4{v[i][0], v[i][1], v[i][2], v[i][3]};
        }
        gg_order();
    }
    // the product of x with the weights at columns c .. c + 3 (c a multiple of 4) after a row's first block
    static __device__ __forceinline__ float four(const u8* row, u32 c, const f32x4& x) {
        const u8* b = row + c / 32 * 34;
        float s = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; i++) s = __builtin_fmaf((float) (i8) b[2 + c % 32 + i], x[i], s);
        return s * f16_to_f32(*(const u16*) b);
    }
    // four codes to f16: 0x6400 | (code ^ 0x80) is 1024 + code + 128
    static __device__ __forceinline__ void codes(u32 v, u32& lo, u32& hi) {
        const u32 t = v ^ 0x80808080u;
        const f16x2 k = {(_Float16) -1152.0f, (_Float16) -1152.0f};
        lo = gg_bits(gg_pair(__builtin_amdgcn_perm(0x64646464u, t, 0x04010400u)) + k);
        hi = gg_bits(gg_pair(__builtin_amdgcn_perm(0x64646464u, t, 0x04030402u)) + k);
    }
    template <int NG>
    __device__ __forceinline__ void products(const u32* strip, const u32x4 (&a)[NG][8], u32 lane, const u32*, float (&out)[NG]) const {
        const u32* row = strip + (lane & 15) * PITCH;
        const u32* own = row + 2 * (lane >> 4);
#pragma unroll
        for (int b = 0; b < 8; b++) {
            {
                // a pair of blocks is 17 words: the even one's codes start in the middle of a word
                const int k = 17 * (b >> 1);
                u32 c0, c1, d;
                if (b & 1) {
                    d = row[k + 8] >> 16;
                    c0 = own[k + 9];
                    c1 = own[k + 10];
                } else {
                    d = row[k] & 0xffffu;
                    const u32 w0 = own[k], w1 = own[k + 1], w2 = own[k + 2];
                    c0 = __builtin_amdgcn_alignbit(w1, w0, 16);
                    c1 = __builtin_amdgcn_alignbit(w2, w1, 16);
                }
                u32 t0, t1, t2, t3;
                codes(c0, t0, t1);
                codes(c1, t2, t3);
                const f16x8 wv = __builtin_bit_cast(f16x8, u32x4{t0, t1, t2, t3});
                const float dd = f16_to_f32((u16) d);
#pragma unroll
                for (int G = 0; G < NG; G++) {
                    const f32x4 s = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a[G][b]), wv, f32x4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
                    out[G] = __builtin_fmaf(gg_sum(s), dd, out[G]);
                }
            }
            if (b & 1) __builtin_amdgcn_sched_barrier(0);   // two blocks' words in registers at a time, not eight
        }
    }
};
// IQ3_S: lane group g takes the sub-blocks 2 g and 2 g + 1 of the 256-block, 64 weights that lie together: the k order of the
// eight matrix instructions is the lane's own (instruction i: columns 64 g + 8 i ..), the same on both operands.
struct GgIq3 {
    static constexpr u32 QK = 256, BB = 110;
    static constexpr bool grid = true, zeros = false;
    static constexpr u32 part_at(u32 q, u32 g) { return 64 * g + 8 * q; }
    u32 qs[4], sg[2], qh, sc, d;
    __device__ __forceinline__ void init(u32) {}
    __device__ __forceinline__ void load(const u8* __restrict__ w, u32 rb, u32 first, u32 rows, u32 col, u32 lane) {
        const u32 g = lane >> 4;
        const u8* p = w + (u64) min(first + (lane & 15), rows - 1) * rb + col / 256 * BB;
        const u32x4b v = *(const u32x4b*) (p + 2 + 16 * g);
        const u32x2b s = *(const u32x2b*) (p + 74 + 8 * g);
#pragma unroll
        for (int i = 0; i < 4; i++) qs[i] = v[i];
        sg[0] = s[0];
        sg[1] = s[1];
        qh = *(const u16*) (p + 66 + 2 * g);
        sc = p[106 + g];
        d = *(const u16*) p;
    }
    __device__ __forceinline__ void stage(u32*, const u8*, u32, u32, u32, u32) const {}
    template <int NG>
    __device__ __forceinline__ void products(const u32*, const u32x4 (&a)[NG][8], u32, const u32* table, float (&out)[NG]) const {
        f32x4 s[NG];
#pragma unroll
        for (int G = 0; G < NG; G++) s[G] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int h = 0; h < 2; h++) {
            // (1024 + magnitude) * scale - 1024 * scale = magnitude * scale, exact and in one packed multiply-add
            const _Float16 sf = (_Float16) (float) (1 + 2 * ((sc >> (4 * h)) & 15u));
            const f16x2 sp = {sf, sf}, sn = {(_Float16) (-1024.0f * (float) sf), (_Float16) (-1024.0f * (float) sf)};
#pragma unroll
            for (int i = 0; i < 4; i++) {
                u32x4 w;
#pragma unroll
                for (int e = 0; e < 2; e++) {
                    const int j = 8 * h + 2 * i + e;   // grid entry of the lane's 16
                    const u32 at = (__builtin_amdgcn_ubfe(qs[j >> 2], 8 * (j & 3), 8) << 2) | (__builtin_amdgcn_ubfe(qh, j, 1) << 10);
                    const u32 m = *(const u32*) ((const u8*) table + at);
                    const u32 n = __builtin_amdgcn_ubfe(sg[j >> 3], 4 * (j & 7), 4);
                    const f16x2 lo = __builtin_elementwise_fma(gg_pair(__builtin_amdgcn_perm(0x64646464u, m, 0x04010400u)), sp, sn);
                    const f16x2 hi = __builtin_elementwise_fma(gg_pair(__builtin_amdgcn_perm(0x64646464u, m, 0x04030402u)), sp, sn);
                    // a set sign bit flips its value's sign: bits 0, 1 to bits 15, 31 of the pair, bits 2, 3 of the other
                    w[2 * e] = gg_bits(lo) ^ ((n * 0x40008000u) & 0x80008000u);
                    w[2 * e + 1] = gg_bits(hi) ^ (((n >> 2) * 0x40008000u) & 0x80008000u);
                }
#pragma unroll
                for (int G = 0; G < NG; G++)
                    s[G] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a[G][4 * h + i]), __builtin_bit_cast(f16x8, w), s[G], 0, 0, 0);
                if (i & 1) __builtin_amdgcn_sched_barrier(0);
            }
        }
        const float dd = f16_to_f32((u16) d);
#pragma unroll
        for (int G = 0; G < NG; G++) out[G] = __builtin_fmaf(gg_sum(s[G]), dd, out[G]);
    }
};

// The bits of the largest magnitude among the chunk's columns of one input (a lane has four): as whole numbers, which order
// like the floats, over the lanes of a row, the rows, and out of the last lane.
template <int ctrl, int rows>
__device__ __forceinline__ u32 gg_max_step(u32 v) { return max(v, (u32) __builtin_amdgcn_update_dpp(0, v, ctrl, rows, 0xf, true)); }
__device__ __forceinline__ u32 gg_most(const f32x4& x) {
    u32 v = f32_bits(fmaxf(fmaxf(__builtin_fabsf(x[0]), __builtin_fabsf(x[1])), fmaxf(__builtin_fabsf(x[2]), __builtin_fabsf(x[3])))) & 0x7fffffffu;
    v = gg_max_step<0x111, 0xf>(v);   // row_shr 1, 2, 4, 8
    v = gg_max_step<0x112, 0xf>(v);
    v = gg_max_step<0x114, 0xf>(v);
    v = gg_max_step<0x118, 0xf>(v);
    v = gg_max_step<0x142, 0xa>(v);   // row_bcast 15, 31
    v = gg_max_step<0x143, 0xc>(v);
    return __builtin_amdgcn_readlane(v, 63);
}

// An input's three parts at a scale, and what they leave of it (in units of the scale, exact like the differences on the way).
__device__ __forceinline__ float gg_parts(float x, float scale, _Float16& p0, _Float16& p1, _Float16& p2) {
    p0 = (_Float16) (x * scale);
    const float r1 = __builtin_fmaf(x, scale, -(float) p0);
    p1 = (_Float16) (r1 * 0x1p11f);
    const float r2 = __builtin_fmaf((float) p1, -0x1p-11f, r1);
    p2 = (_Float16) (r2 * 0x1p22f);
    return __builtin_fmaf((float) p2, -0x1p-22f, r2);
}

// 256 columns of the inputs 4 G .. 4 G + 3 (v[r]: the lane's four columns of each), as the lane's operand registers: the three
// parts of the n that there are go through the strip (the rows of others hold what lay there: their sums go nowhere).  iv undoes
// the scale of input 4 G + lane / 16.  Returns whether the parts are not all of some input (which is then under 2^-37 times the
// largest).
template <class F>
__device__ __forceinline__ bool gg_split(const f32x4 (&v)[4], u32 n, u32* strip, u32 lane, u32x4 (&a)[8], float& iv) {
    u16* st = (u16*) strip;
    u32 rest = 0;
    iv = 1.0f;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        if ((u32) r < n) {
            u32 part[3][2];
            const u32 mx = gg_most(v[r]);
            float scale, inv;
            pow2_scale_of(mx, scale, inv);
            if (lane >> 4 == (u32) r) iv = inv;
            // an infinity is all in its first part: what it leaves would be a NaN
            const u32 keep = mx == 0x7f800000u ? 0u : ~0u;
#pragma unroll
            for (int i = 0; i < 2; i++) {
                _Float16 t[2][3];
#pragma unroll
                for (int e = 0; e < 2; e++) rest |= f32_bits(gg_parts(v[r][2 * i + e], scale, t[e][0], t[e][1], t[e][2]));
                part[0][i] = gg_bits(f16x2{t[0][0], t[1][0]});
                part[1][i] = gg_bits(f16x2{t[0][1], t[1][1]}) & keep;
                part[2][i] = gg_bits(f16x2{t[0][2], t[1][2]}) & keep;
            }
#pragma unroll
            for (int p = 0; p < 3; p++) *(uint2*) (st + (3 * r + p) * GG_PITCH + 4 * lane) = uint2{part[p][0], part[p][1]};
        }
    }
    gg_order();
    const u32 ar = lane & 15;
    const u16* rowp = st + ((ar >> 2) * 3 + min(ar & 3, 2u)) * GG_PITCH;
#pragma unroll
    for (u32 q = 0; q < 8; q++) a[q] = *(const u32x4*) (rowp + F::part_at(q, lane >> 4));
    gg_order();
    return F::zeros && __builtin_amdgcn_ballot_w64(rest != 0) != 0;
}

// Sixteen rows of a matrix.
struct GgTile {
    const u8* w;
    u32 first;
};

// The products of what the three parts leave of a chunk's inputs, on the vector unit and a row at a time, into the sums of the
// workgroup's tiles: rare, so short rather than fast.  col: the lane's four columns, if they are `mine` to add; off: from a row's
// first byte to the chunk's first block.
template <class F, int NG, class Tile, class Input>
__device__ __forceinline__ void gg_rest(Tile tile, u32 off, u32 rb, u32 rows, u32 nt, Input input, u32 col, u32 m, bool mine, u32 lane, float* tot) {
#pragma unroll 1
    for (u32 j = 0; j < m; j++) {
        f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
        if (mine) v = *(const f32x4*) (input(j) + col);
        float scale, inv;
        const u32 mx = gg_most(v);
        if (mx >= 0x7f800000u) continue;   // nothing finite comes of it
        pow2_scale_of(mx, scale, inv);
        bool any = false;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            _Float16 p0, p1, p2;
            v[i] = gg_parts(v[i], scale, p0, p1, p2);
            any = any || v[i] != 0.0f;
        }
        if (!__builtin_amdgcn_ballot_w64(any)) continue;
#pragma unroll 1
        for (u32 i = 0; i < 16 * nt; i++) {
            const GgTile t = tile(i / 16);
            const u32 row = t.first + i % 16;
            float s = mine && row < rows ? F::four(t.w + (u64) row * rb + off, 4 * lane, v) : 0.0f;
            s = seg_sum<64>(s, lane);
            float* at = tot + (i / 16 * NG + j / 4) * 64;
            if (lane == 16 * (j & 3) + i % 16) *at = __builtin_fmaf(s, inv, *at);
        }
    }
}

extern __shared__ __attribute__((aligned(16))) u32 sz_dyn_lds[];

// The sums of a workgroup: nt tiles of 16 rows (tile(t): the matrix and the first of the 16) for m inputs of `cols`
// columns (input(j): its first).  Its W waves take the chunks w, w + W, .. of the row (W by the number of chunks alone: the sums'
// order, so the bits, do not depend on m).  A row's last chunk, where it is short, is its last 256 columns, the inputs of the ones
// that the chunk before has taken as zeros.  Ends with the waves' sums in LDS behind a barrier; gg_total adds them up.
// Dynamic LDS: GG_STRIP and nt * NG * 64 words a wave; table: 512 words of a format with a grid.
template <class F, int NG, class Tile, class Input>
__device__ __forceinline__ void gg_sums(Tile tile, u32 nt, u32 rows, Input input, u32 m, u32 cols, u32* table) {
    const u32 wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, W = blockDim.x >> 6;
    const u32 rb = cols / F::QK * F::BB, nc = (cols + 255) / 256;
    u32* strip = sz_dyn_lds + wave * GG_STRIP;
    float* tot = (float*) (sz_dyn_lds + W * GG_STRIP) + wave * (nt * NG * 64) + lane;   // [wave][tile][G][lane]: a lane adds to its own places
    auto start = [&](u32 c) { return cols < 256 ? 0u : min(256 * c, cols - 256); };
    F cur;
    cur.init(lane);
    for (u32 t = 0; t < nt * NG; t++) tot[64 * t] = 0.0f;
    bool left = false;
    for (u32 c = wave; c < nc; c += W) {
        const u32 col = start(c) + 4 * lane;
        f32x4 v[NG][4];
#pragma unroll
        for (int r = 0; r < 4 * NG; r++) {
            v[r >> 2][r & 3] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            if ((u32) r < m && col >= 256 * c && col < cols) v[r >> 2][r & 3] = *(const f32x4*) (input(r) + col);
        }
        if (c == wave) {
            const GgTile t0 = tile(0);
            cur.load(t0.w, rb, t0.first, rows, start(c), lane);   // W <= nc
            if constexpr (F::grid) {
                for (u32 i = threadIdx.x; i < 512; i += blockDim.x) table[i] = IQ3S_GRID[i];
                __syncthreads();
            }
        }
        u32x4 a[NG][8];
        float iv[NG];
#pragma unroll
        for (int G = 0; G < NG; G++) left = gg_split<F>(v[G], m - min(m, 4u * G), strip, lane, a[G], iv[G]) || left;
#pragma unroll 1
        for (u32 t = 0; t < nt; t++) {
            const GgTile tt = tile(t);
            F now = cur;
            now.stage(strip, tt.w, rb, tt.first, rows, lane);
            if (t + 1 < nt || c + W < nc) {
                const GgTile next = tile(t + 1 < nt ? t + 1 : 0);
                cur.load(next.w, rb, next.first, rows, start(t + 1 < nt ? c : c + W), lane);
            }
            float out[NG];
#pragma unroll
            for (int G = 0; G < NG; G++) out[G] = 0.0f;
            now.template products<NG>(strip, a, lane, table, out);
#pragma unroll
            for (int G = 0; G < NG; G++) tot[(t * NG + G) * 64] = __builtin_fmaf(out[G], iv[G], tot[(t * NG + G) * 64]);
            gg_order();   // the strip is read before the next tile goes there (LDS is in order within a wave)
        }
    }
    if constexpr (F::zeros) {
        if (left)
            for (u32 c = wave; c < nc; c += W) {
                const u32 col = start(c) + 4 * lane;
                gg_rest<F, NG>(tile, start(c) / F::QK * F::BB, rb, rows, nt, input, col, m, col >= 256 * c && col < cols, lane, tot);
            }
    }
    __syncthreads();
}
// Place i (tile * NG + G) * 64 + lane of the sums: row lane % 16 of the tile, input 4 G + lane / 16.
template <int NG>
__device__ __forceinline__ float gg_total(u32 i, u32 nt) {
    const u32 W = blockDim.x >> 6;
    const float* sums = (const float*) (sz_dyn_lds + W * GG_STRIP);
    float s = sums[i];
    for (u32 k = 1; k < W; k++) s += sums[k * (nt * NG * 64) + i];
    return s;
}

// y_j = W x_j, j < m: x rows xs floats apart, y rows ys apart (matvec_cols_*, kernels/matvec.cu:677).  A workgroup takes the
// tiles blockIdx.x, blockIdx.x + gridDim.x, .. of 16 rows (at most 4).  block 64 W, at most 1024.
template <class F, int NG>
__device__ __forceinline__ void gg_cols(const u8* __restrict__ w, const float* __restrict__ x, u32 xs, float* __restrict__ y, u32 ys, u32 rows, u32 cols, u32 m) {
    __shared__ u32 table[F::grid ? 512 : 1];
    const u32 n16 = (rows + 15) / 16, nt = (n16 - blockIdx.x + gridDim.x - 1) / gridDim.x;
    gg_sums<F, NG>([&](u32 t) { return GgTile{w, 16 * (blockIdx.x + t * gridDim.x)}; }, nt, rows, [&](u32 j) { return x + (u64) j * xs; }, m, cols, table);
    for (u32 i = threadIdx.x; i < nt * NG * 64; i += blockDim.x) {
        const u32 t = i / (NG * 64), G = i / 64 % NG, l = i & 63;
        const u32 r = 16 * (blockIdx.x + t * gridDim.x) + (l & 15), j = 4 * G + (l >> 4);
        if (r < rows && j < m) y[(u64) j * ys + r] = gg_total<NG>(i, nt);
    }
}
extern "C" __global__ void __launch_bounds__(1024, 4) matvec_cols_q8_0(const u8* w, const float* x, u32 xs, float* y, u32 ys, u32 rows, u32 cols, u32 m) {
    gg_cols<GgQ8, 1>(w, x, xs, y, ys, rows, cols, m);
}
extern "C" __global__ void __launch_bounds__(1024, 4) matvec_cols_w_q8_0(const u8* w, const float* x, u32 xs, float* y, u32 ys, u32 rows, u32 cols, u32 m) {
    gg_cols<GgQ8, 2>(w, x, xs, y, ys, rows, cols, m);
}
extern "C" __global__ void __launch_bounds__(1024, 4) matvec_cols_iq3_s(const u8* w, const float* x, u32 xs, float* y, u32 ys, u32 rows, u32 cols, u32 m) {
    gg_cols<GgIq3, 1>(w, x, xs, y, ys, rows, cols, m);
}
extern "C" __global__ void __launch_bounds__(1024, 4) matvec_cols_w_iq3_s(const u8* w, const float* x, u32 xs, float* y, u32 ys, u32 rows, u32 cols, u32 m) {
    gg_cols<GgIq3, 2>(w, x, xs, y, ys, rows, cols, m);
}

// ------------------------------------------------------------------------------------- MoE layers, by distinct expert
// The verify layer of GGUF experts for one to eight tokens, on the products above: every distinct expert's weights are decoded once for
// the tokens that chose it (route_plan in route.hip.h lists them).  Expert e's gate, up and down lie at experts + e stride + {0, part,
// 2 part}, the shared one's at shared + the same.  A workgroup takes 2 to 8 row tiles of one expert (the host's choice), a wave a
// 256-column chunk; the first launch has the same rows of gate and up and leaves silu(gate) * up.  Measured, 8 tokens of top-8 of 128
// Q8_0 experts of 2560 x 768 (52 distinct): 49 us (4.4 TB/s) and 23 us (4.7 TB/s), where the vector unit took 110 and 50 pair by
// pair: bound by the weights' way from memory.  The same layers of IQ3_S experts take 91 us (148), bound by the decode and its table
// look-ups.  Requesting the inputs ahead of a pair's selection kept values across it in registers (78 -> 113) and lost 3 to 6 %.
template <int N>
struct GgInt {
    static constexpr int value = N;
};
// An item of the plan: its expert's first byte, its tokens' rows and pair numbers.
struct GgItem {
    const u8* w;
    u32 n;
    u64 toks, pairs[2];
    __device__ __forceinline__ u32 token(u32 r) const { return (u32) (toks >> (8 * r)) & 0xffu; }
    __device__ __forceinline__ u32 pair(u32 r) const { return (u32) ((r < 4 ? pairs[0] : pairs[1]) >> (16 * (r & 3))) & 0xffffu; }
};
__device__ __forceinline__ u64 gg_uniform(u32 lo, u32 hi) { return (u64) (u32) __builtin_amdgcn_readfirstlane(lo) | ((u64) (u32) __builtin_amdgcn_readfirstlane(hi) << 32); }
// Item `it` of the launch, if there is one.  ioff = 0: there is no plan; the items are the shared expert with all m tokens (0) and then
// the (token, rank) pairs, whose expert select(pair) gives.  A token's sums do not depend on the other tokens of its item: both forms
// give the same bits.
template <class Select>
__device__ __forceinline__ bool gg_item(const u8* __restrict__ pbuf, u32 ioff, u32 it, u64 experts, u64 stride, u64 shared, u32 k, u32 m, Select select, GgItem& item) {
    u32 e = 0xffffffffu;
    if (ioff) {
        const u32* plan = (const u32*) (pbuf + ioff);
        const u32x4 lo = *(const u32x4*) (plan + 4 + 8 * it), hi = *(const u32x4*) (plan + 8 + 8 * it);   // there for every slot, an item or not
        if (it >= plan[0]) return false;
        e = __builtin_amdgcn_readfirstlane(lo[0]);
        item.n = __builtin_amdgcn_readfirstlane(lo[1]);
        item.toks = gg_uniform(lo[2], lo[3]);
        item.pairs[0] = gg_uniform(hi[0], hi[1]);
        item.pairs[1] = gg_uniform(hi[2], hi[3]);
    } else if (it > 0) {
        e = __builtin_amdgcn_readfirstlane(select(it - 1));
        if (e == 0xffffffffu) return false;
        item.n = 1;
        item.toks = (it - 1) / k;
        item.pairs[0] = it - 1;
        item.pairs[1] = 0;
    } else {
        if (!shared) return false;
        const u64 ones = 0x0001000100010001ull, first = 0x0003000200010000ull + ones * (m * k);
        item.n = m;
        item.toks = 0x0706050403020100ull;
        item.pairs[0] = first;
        item.pairs[1] = first + 4 * ones;
    }
    item.w = (const u8*) (e == 0xffffffffu ? shared : experts + e * stride);
    return true;
}

// The routing weights and counts of the chosen experts, by a workgroup that has nothing else to do.
__device__ __forceinline__ void gg_route_weights(const float* __restrict__ logits, u8* __restrict__ pbuf, u32 ne, u32 k, u32 m) {
    const u32 lane = threadIdx.x & 63;
    for (u32 j = threadIdx.x >> 6; j < m; j += blockDim.x >> 6) {
        u32 kk;
        const float wt = route_weights(logits + (u64) j * ne, ne, k, lane, (const u32*) pbuf + j * k, &kk);
        if (lane < k) ((float*) (pbuf + m * k * 4))[j * k + lane] = wt;
        if (lane == 0) ((u32*) (pbuf + 2 * m * k * 4))[j] = kk;
    }
}

// Launch 2 (the plan is launch 1): act[pair][ff] = silu(gate) * up.  grid = (workgroups a projection, slots = m k + 2:
// the last is never an item and has the routing weights and counts worked out instead), block 64 W as for gg_sums.
// Without a plan (slots = m k + 1) a workgroup selects its pair's expert on one of its waves and launch 3 works the weights out.
template <class F, int NG>
__device__ __forceinline__ void gg_gate_up(const float* __restrict__ logits, u64 experts, u64 stride, u64 shared, u32 part, u8* __restrict__ pbuf, u32 ioff, const float* __restrict__ u,
                                           float* __restrict__ act, u32 ne, u32 k, u32 m, u32 hidden, u32 ff) {
    __shared__ u32 table[F::grid ? 512 : 1];
    __shared__ u32 top[16];
    const u32 lane = threadIdx.x & 63;
    if (ioff && blockIdx.y == gridDim.y - 1) {
        if (blockIdx.x == 0) gg_route_weights(logits, pbuf, ne, k, m);
        return;
    }
    GgItem it;
    auto select = [&](u32 pair) {
        const u32 j = pair / k, t = pair - j * k;
        if (threadIdx.x < 64) {
            __builtin_amdgcn_s_setprio(3);   // every other wave of the workgroup waits for this one
            route_id_of_rank(logits + (u64) j * ne, ne, k, t, lane, (double*) sz_dyn_lds, top);   // only top[t] is read
            __builtin_amdgcn_s_setprio(0);
            if (blockIdx.x == 0 && lane == 0) ((u32*) pbuf)[pair] = top[t];
        }
        __syncthreads();
        return top[t];
    };
    if (!gg_item(pbuf, ioff, blockIdx.y, experts, stride, shared, k, m, select, it)) return;
    const u32 n16 = ff / 16, nt = (n16 - blockIdx.x + gridDim.x - 1) / gridDim.x;
    auto run = [&](auto ng) {
        constexpr int N = decltype(ng)::value;
        gg_sums<F, N>([&](u32 t) { return GgTile{it.w + (t & 1 ? part : 0u), 16 * (blockIdx.x + (t >> 1) * gridDim.x)}; }, 2 * nt, ff,
                      [&](u32 r) { return u + (u64) it.token(r) * hidden; }, it.n, hidden, table);
        for (u32 i = threadIdx.x; i < nt * N * 64; i += blockDim.x) {
            const u32 t = i / (N * 64), l = i % (N * 64), r = l >> 4;
            if (r >= it.n) continue;
            const float g = gg_total<N>(2 * t * N * 64 + l, 2 * nt), up = gg_total<N>((2 * t + 1) * N * 64 + l, 2 * nt);
            act[(u64) it.pair(r) * ff + 16 * (blockIdx.x + t * gridDim.x) + (l & 15)] = siluf_ref(g) * up;
        }
    };
    if constexpr (NG > 1) {
        if (it.n > 4) return run(GgInt<NG>());
    }
    run(GgInt<1>());
}

// Launch 3: eo[pair][hidden] = down act.  grid = (workgroups, slots = m k + 1, or without a plan m k + 2, the last one for the
// weights), block as for gg_sums.
template <class F, int NG>
__device__ __forceinline__ void gg_down(const float* __restrict__ logits, u64 experts, u64 stride, u64 shared, u32 part, u8* __restrict__ pbuf, u32 ioff, const float* __restrict__ act,
                                        float* __restrict__ eo, u32 ne, u32 k, u32 m, u32 hidden, u32 ff) {
    __shared__ u32 table[F::grid ? 512 : 1];
    if (!ioff && blockIdx.y == gridDim.y - 1) {
        if (blockIdx.x == 0) gg_route_weights(logits, pbuf, ne, k, m);
        return;
    }
    GgItem it;
    if (!gg_item(pbuf, ioff, blockIdx.y, experts, stride, shared, k, m, [&](u32 pair) { return ((const u32*) pbuf)[pair]; }, it)) return;
    const u32 n16 = hidden / 16, nt = (n16 - blockIdx.x + gridDim.x - 1) / gridDim.x;
    auto run = [&](auto ng) {
        constexpr int N = decltype(ng)::value;
        gg_sums<F, N>([&](u32 t) { return GgTile{it.w + 2 * (u64) part, 16 * (blockIdx.x + t * gridDim.x)}; }, nt, hidden,
                      [&](u32 r) { return act + (u64) it.pair(r) * ff; }, it.n, ff, table);
        for (u32 i = threadIdx.x; i < nt * N * 64; i += blockDim.x) {
            const u32 t = i / (N * 64), l = i % (N * 64), r = l >> 4;
            if (r < it.n) eo[(u64) it.pair(r) * hidden + 16 * (blockIdx.x + t * gridDim.x) + (l & 15)] = gg_total<N>(i, nt);
        }
    };
    if constexpr (NG > 1) {
        if (it.n > 4) return run(GgInt<NG>());
    }
    run(GgInt<1>());
}
extern "C" __global__ void __launch_bounds__(1024, 4) verify_items_gate_up_q8_0(const float* logits, u64 experts, u64 stride, u64 shared, u32 part, u8* pbuf, u32 ioff, const float* u, float* act,
                                                                              u32 ne, u32 k, u32 m, u32 hidden, u32 ff) {
    gg_gate_up<GgQ8, 1>(logits, experts, stride, shared, part, pbuf, ioff, u, act, ne, k, m, hidden, ff);
}
extern "C" __global__ void __launch_bounds__(1024, 4) verify_items_down_q8_0(const float* logits, u64 experts, u64 stride, u64 shared, u32 part, u8* pbuf, u32 ioff, const float* act, float* eo, u32 ne, u32 k,
                                                                           u32 m, u32 hidden, u32 ff) {
    gg_down<GgQ8, 1>(logits, experts, stride, shared, part, pbuf, ioff, act, eo, ne, k, m, hidden, ff);
}
extern "C" __global__ void __launch_bounds__(1024, 4) verify_items_gate_up_w_q8_0(const float* logits, u64 experts, u64 stride, u64 shared, u32 part, u8* pbuf, u32 ioff, const float* u, float* act,
                                                                              u32 ne, u32 k, u32 m, u32 hidden, u32 ff) {
    gg_gate_up<GgQ8, 2>(logits, experts, stride, shared, part, pbuf, ioff, u, act, ne, k, m, hidden, ff);
}
extern "C" __global__ void __launch_bounds__(1024, 4) verify_items_down_w_q8_0(const float* logits, u64 experts, u64 stride, u64 shared, u32 part, u8* pbuf, u32 ioff, const float* act, float* eo, u32 ne, u32 k,
                                                                           u32 m, u32 hidden, u32 ff) {
    gg_down<GgQ8, 2>(logits, experts, stride, shared, part, pbuf, ioff, act, eo, ne, k, m, hidden, ff);
}
extern "C" __global__ void __launch_bounds__(1024, 4) verify_items_gate_up_iq3_s(const float* logits, u64 experts, u64 stride, u64 shared, u32 part, u8* pbuf, u32 ioff, const float* u, float* act,
                                                                              u32 ne, u32 k, u32 m, u32 hidden, u32 ff) {
    gg_gate_up<GgIq3, 1>(logits, experts, stride, shared, part, pbuf, ioff, u, act, ne, k, m, hidden, ff);
}
extern "C" __global__ void __launch_bounds__(1024, 4) verify_items_down_iq3_s(const float* logits, u64 experts, u64 stride, u64 shared, u32 part, u8* pbuf, u32 ioff, const float* act, float* eo, u32 ne, u32 k,
                                                                           u32 m, u32 hidden, u32 ff) {
    gg_down<GgIq3, 1>(logits, experts, stride, shared, part, pbuf, ioff, act, eo, ne, k, m, hidden, ff);
}
extern "C" __global__ void __launch_bounds__(1024, 4) verify_items_gate_up_w_iq3_s(const float* logits, u64 experts, u64 stride, u64 shared, u32 part, u8* pbuf, u32 ioff, const float* u, float* act,
                                                                              u32 ne, u32 k, u32 m, u32 hidden, u32 ff) {
    gg_gate_up<GgIq3, 2>(logits, experts, stride, shared, part, pbuf, ioff, u, act, ne, k, m, hidden, ff);
}
extern "C" __global__ void __launch_bounds__(1024, 4) verify_items_down_w_iq3_s(const float* logits, u64 experts, u64 stride, u64 shared, u32 part, u8* pbuf, u32 ioff, const float* act, float* eo, u32 ne, u32 k,
                                                                           u32 m, u32 hidden, u32 ff) {
    gg_down<GgIq3, 2>(logits, experts, stride, shared, part, pbuf, ioff, act, eo, ne, k, m, hidden, ff);
}

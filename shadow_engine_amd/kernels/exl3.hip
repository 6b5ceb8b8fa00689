// EXL3 (trellis-coded, Hadamard-rotated) matrix-vector products for 1..8 inputs, bit rates K = 1..8 and K + 1/2 (K = 1..3), codebook
// "mul1".  Format and arithmetic follow the CPU reference (crates/shadowzero-model/src/exl3.rs): a projection is a blob
// [suh f16[in] | svh f16[out] | 4-byte marker | trellis], the trellis is [in/16][out/16] tiles of 16 K u16 words, a tile is
// a ring of 256 K bits (most significant bit first inside little-endian u32 words) and weight t's 16-bit state ends at
// bit (t + 1) K; y = ((x * suh) H) W_hat H * svh with H the 128-point Walsh-Hadamard transform over 128-blocks.
//
// Lane map (wave64, made for this format rather than taken from the 32-lane tensor-core order the trellis was laid out
// for): one wave decodes the 8 tiles of one tile row of a 128-output block, which are 256 K contiguous bytes.  Lane
// L = 8 c + q takes weights 32 q .. 32 q + 31 of tile c: exactly K consecutive u32 words of the ring plus the word before
// them for the first windows, so every window position is a compile-time constant.  By the tile's position map
// (exl3.rs:106) those 32 weights are all 16 input rows of output columns q and q + 8 of the tile, so a lane owns two
// output columns outright and no cross-lane sum is needed inside a tile row.

__device__ __forceinline__ _Float16 exl3_cb2(u32 state) {
    // exl3.rs:87-94: the byte sum of state * 0x83DCD12D on top of 0x6400 is an f16 in [1024, 2048); one fused f16 multiply-add
    const u32 x = state * 0x83DCD12Du;
    const u32 s = __builtin_amdgcn_sad_u8(x, 0u, 0x6400u);
    const _Float16 h = __builtin_bit_cast(_Float16, (u16) s);
    return __builtin_fmaf16(h, __builtin_bit_cast(_Float16, (u16) 0x1eee), __builtin_bit_cast(_Float16, (u16) 0xc931));
}

// All 65,536 codebook values as f32 (crates/shadowzero-cuda/tests/exl3.rs:65-77 checks them bit for bit).
extern "C" __global__ void __launch_bounds__(256) exl3_codebook(float* out, u32 n) {
    const u32 i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) out[i] = (float) exl3_cb2(i);
}

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

// state * 0x83DCD12D modulo 2^32: one v_mul_lo_u32, which issues at the full vector rate on this chip (measured: the same
// rate as the 24-bit multiply and the byte-sum instruction).
__device__ __forceinline__ u32 exl3_mul(u32 state) { return state * 0x83DCD12Du; }

// Two states to their two f16 weights at once: both byte sums land in one register as a pair of f16 bit patterns
// (v_sad_u8 into the low half, v_sad_hi_u8 into the high half, each on top of 0x6400), then one packed fused multiply-add.
// The same arithmetic per weight as exl3_cb2.
__device__ __forceinline__ f16x2 exl3_cb2_pair(u32 sa, u32 sb) {
    const u32 lo = __builtin_amdgcn_sad_u8(exl3_mul(sa), 0u, 0x64006400u);
    const u32 both = __builtin_amdgcn_sad_hi_u8(exl3_mul(sb), 0u, lo);
    const f16x2 h = __builtin_bit_cast(f16x2, both);
    const f16x2 kinv = {__builtin_bit_cast(_Float16, (u16) 0x1eee), __builtin_bit_cast(_Float16, (u16) 0x1eee)};
    const f16x2 kbias = {__builtin_bit_cast(_Float16, (u16) 0xc931), __builtin_bit_cast(_Float16, (u16) 0xc931)};
    return __builtin_elementwise_fma(h, kinv, kbias);
}

// Bit rates: K bits a weight, or K + 1/2 (H: positions alternate K and K + 1 bits, a pair takes 2 K + 1; exl3.rs:164).  A lane
// decodes 32 consecutive weights = EXL3_LANE_BITS stream bits; with a half rate that is an odd number of 16-bit halves, so
// every second lane of a tile starts in the middle of a word.
#define EXL3_LANE_BITS(K, H) (16 * (2 * (K) + (H)))          /* stream bits of a lane's 32 weights */
#define EXL3_TILE_WORDS(K, H) (4 * (2 * (K) + (H)))          /* u32 words of a tile's ring: 8 K, or 4 (2 K + 1) */
#define EXL3_NW(K, H) ((K) + 1 + (H))                        /* words S[] of a lane: the 32 stream bits before its own, then its own */

// End of the window of the lane's weight i, in stream bits after the lane's first own bit (Rate::end_bit, exl3.rs:164).
template <int K, bool H>
__device__ __forceinline__ constexpr int exl3_end(int i) {
    return H ? (i >> 1) * (2 * K + 1) + ((i & 1) ? 2 * K + 1 : K) : (i + 1) * K;
}

// The state of the lane's weight i from S = the stream from 32 bits before the lane's own bits on (S[0] = the ring word
// before its own for an integer rate), and T = the same stream 16 bits on (T[n] = stream bits [32 n + 16, 32 n + 48)), so
// that every window lies inside one register.
template <int K, bool H = false>
__device__ __forceinline__ u32 exl3_state(const u32 (&S)[EXL3_NW(K, H)], const u32 (&T)[EXL3_NW(K, H) - 1], int i) {
    const int a = 16 + exl3_end<K, H>(i);   // first stream bit of the window, counted from the first bit of S[0]
    const int n = a / 32, r = a % 32;
    return r <= 16 ? __builtin_amdgcn_ubfe(S[n], 16 - r, 16) : __builtin_amdgcn_ubfe(T[n], 32 - r, 16);
}

// The 32 weights of a lane, as 16 pairs (weights 2 p and 2 p + 1).
template <int K, bool H = false>
__device__ __forceinline__ void exl3_decode32(const u32 (&S)[EXL3_NW(K, H)], f16x2 (&w)[16]) {
    u32 T[EXL3_NW(K, H) - 1];
#pragma unroll
    for (int n = 0; n < EXL3_NW(K, H) - 1; n++) T[n] = __builtin_amdgcn_alignbit(S[n], S[n + 1], 16);
#pragma unroll
    for (int p = 0; p < 16; p++) w[p] = exl3_cb2_pair(exl3_state<K, H>(S, T, 2 * p), exl3_state<K, H>(S, T, 2 * p + 1));
}

// Input row (0..15) and output-column half (0: column q, 1: column q + 8) of a lane's weight i.
#define EXL3_ROW(i) (2 * ((i) >> 3) + ((i) & 1) + 8 * (((i) >> 1) & 1))
#define EXL3_HALF(i) (((i) >> 2) & 1)

// The lane's words S[] of tile (kt, tile column 8 ob + c): `tr` is the trellis as u32 words, nt = out / 16.  Integer rate: the
// lane's own K words are one contiguous 4 K-byte load; the word before them wraps to the tile's last word for the first lane.
// Half rate: lane q's bits start q (16 K + 8) bits into the ring, in the middle of a word for odd q; it reads the words that
// hold the 32 bits before them and its own (cyclically) and, for odd q, shifts the lot by 16 bits.
template <int K, bool H = false>
__device__ __forceinline__ void exl3_load_words(const u32* __restrict__ tr, u32 nt, u32 kt, u32 ob, u32 lane, u32 (&S)[EXL3_NW(K, H)]) {
    const u32 c = lane >> 3, q = lane & 7;
    const u32* tile = tr + ((u64) kt * nt + ob * 8 + c) * EXL3_TILE_WORDS(K, H);
    if constexpr (H) {
        constexpr u32 RW = EXL3_TILE_WORDS(K, H), NW = EXL3_NW(K, H);
        const u32 odd = q & 1;
        const u32 first = q * EXL3_LANE_BITS(K, H) - 16 * odd;    // a multiple of 32: the word that holds the lane's first own bit
        const u32 w0 = first / 32 + RW - 1;                        // one word before it (cyclic)
        u32 L[NW + 1];
#pragma unroll
        for (u32 n = 0; n <= NW; n++) L[n] = tile[(w0 + n) % RW];
#pragma unroll
        for (u32 n = 0; n < NW; n++) S[n] = odd ? __builtin_amdgcn_alignbit(L[n], L[n + 1], 16) : L[n];
    } else {
        S[0] = tile[q == 0 ? 8 * K - 1 : q * K - 1];
        typedef u32 vec __attribute__((ext_vector_type(K), aligned(4)));
        if constexpr (K == 1) {
            S[1] = tile[q];
        } else {
            const vec v = *(const vec*) (tile + q * K);
#pragma unroll
            for (int d = 0; d < K; d++) S[d + 1] = v[d];
        }
    }
}

// W_hat[in][out] as f32, straight from the trellis (exl3.rs:242-256): the bit-exact decode hook.
// grid = (out / 128, in / 16), block 64.
template <int K, bool H = false>
__device__ __forceinline__ void exl3_decode_kernel(const u8* blob, float* what, u32 in_f, u32 out_f) {
    const u32 lane = threadIdx.x, ob = blockIdx.x, kt = blockIdx.y;
    const u32* tr = (const u32*) (blob + 2 * (u64) in_f + 2 * (u64) out_f + 4);
    u32 S[EXL3_NW(K, H)];
    exl3_load_words<K, H>(tr, out_f / 16, kt, ob, lane, S);
    f16x2 w[16];
    exl3_decode32<K, H>(S, w);
    const u32 col = ob * 128 + (lane >> 3) * 16 + (lane & 7);
#pragma unroll
    for (int i = 0; i < 32; i++) what[(u64) (kt * 16 + EXL3_ROW(i)) * out_f + col + 8 * EXL3_HALF(i)] = (float) w[i / 2][i % 2];
}

#define EXL3_ENTRIES(K)                                                                                                              \
    extern "C" __global__ void __launch_bounds__(64) exl3_decode_##K(const u8* blob, float* what, u32 in_f, u32 out_f) {             \
        exl3_decode_kernel<K>(blob, what, in_f, out_f);                                                                              \
    }
#define EXL3_HALF_ENTRIES(K)                                                                                                         \
    extern "C" __global__ void __launch_bounds__(64) exl3_decode_h##K(const u8* blob, float* what, u32 in_f, u32 out_f) {            \
        exl3_decode_kernel<K, true>(blob, what, in_f, out_f);                                                                        \
    }
EXL3_ENTRIES(1)
EXL3_ENTRIES(2)
EXL3_ENTRIES(3)
EXL3_ENTRIES(4)
EXL3_ENTRIES(5)
EXL3_ENTRIES(6)
EXL3_ENTRIES(7)
EXL3_ENTRIES(8)
EXL3_HALF_ENTRIES(1)
EXL3_HALF_ENTRIES(2)
EXL3_HALF_ENTRIES(3)

template <int h>
__device__ __forceinline__ void wht_stage(float& v0, float& v1, u32 lane) {
    const float p0 = lane_xor<h>(v0, lane), p1 = lane_xor<h>(v1, lane);
    // partner - own in the upper lane of a pair, own + partner in the lower: one multiply-add by -1 or +1 (exact)
    const float sgn = bits_f32(0x3f800000u | ((lane & h) ? 0x80000000u : 0u));
    v0 = __builtin_fmaf(v0, sgn, p0);
    v1 = __builtin_fmaf(v1, sgn, p1);
}

// 128-point Walsh-Hadamard transform inside one wave: the lane holds elements `lane` (v0) and `lane + 64` (v1).  Stages
// h = 1, 2, .. 32 cross lanes, h = 64 is the lane's own pair; then the 1/sqrt(128) factor (exl3.rs:583-599), which the
// raw form leaves out.
__device__ __forceinline__ void wht128_wave_raw(float& v0, float& v1, u32 lane) {
    wht_stage<1>(v0, v1, lane);
    wht_stage<2>(v0, v1, lane);
    wht_stage<4>(v0, v1, lane);
    wht_stage<8>(v0, v1, lane);
    wht_stage<16>(v0, v1, lane);
    wht_stage<32>(v0, v1, lane);
    const float a = v0 + v1, b = v0 - v1;
    v0 = a;
    v1 = b;
}

__device__ __forceinline__ void wht128_wave(float& v0, float& v1, u32 lane) {
    wht128_wave_raw(v0, v1, lane);
    v0 *= 0.08838835f;
    v1 *= 0.08838835f;
}

// ------------------------------------------------------------------------------------------- the verify layer
// Resident EXL3 layers for a verify batch (m <= 8 rows): a plan, gate and up, down, the rank-order sum, each launch for one
// layer (sz_moe_layer_verify, sz_moe_block_verify) or for all layers of one type of a round at once (sz_verify_round is
// given every layer's inputs before the first one runs, so the layers do not wait for each other): with 48 layers in a
// launch the two decode launches are bound by the vector unit and not by 96 prologues, tails and launch boundaries.
//
// (1) The work items are the DISTINCT experts of a layer's batch, the shared expert as the first item with all tokens: an
// expert's weights are decoded once however many tokens chose it (at 4 rows and top-10 of 512 experts 40 items for 44
// (token, expert) pairs, at 8 rows 75 for 88, of 32 experts 29 for 72).
// (2) The products run on the matrix cores: a lane decodes 4 consecutive weights of the bit stream, which are four values of
// operand B of v_mfma_f32_16x16x32_f16 as decoded (two tile rows make one instruction), 15 vector instructions a 16 x 16
// tile for up to 4 tokens where the vector unit alone needs 19 a token.  The item's tokens ride on the rows of operand A in
// THREE f16 parts of 11 bits, scaled by the power of two that takes the largest magnitude of the token's 512 inputs to
// [2^14, 2^15), the second and third part 2^11 and 2^22 times more: all 24 bits of an f32 down to 2^-37 of that largest, and an
// error under 2^-61 of it below.  No codebook weight is smaller than 2^-10, so f32 inputs would lose as much in the f32 sums
// that the largest input is part of.  Products are exact and sums are f32, as with f32 inputs.  (An infinite input gives no
// finite output: the transform spreads it over 128 inputs of either sign.)
// (3) A workgroup prepares the A rows of its 512 inputs once (a wave a 128-block: scales, transform, split) and its four
// waves then take CT column tiles each over all 512 inputs, so there is no sum over waves.  The sums are left as they are:
// whoever reads them (launch 2 for gate and up, the last launch for down) adds the partials of the 512-input blocks up and
// applies the output side once.
//
// A layer's table entry: where its experts lie (expert e's gate, up and down at experts + e stride + {0, part, 2 part},
// the shared expert's at shared + the same; shared = 0: none) and its number in the caller's buffers.
struct VerifyLayer {
    u64 experts, stride, shared;
    u32 part, layer;
};
// Layer li of a launch: out of the table, or of a one-layer launch its kernel arguments (table 0): a load less ahead of
// everything else.
__device__ __forceinline__ VerifyLayer verify_layer(const u8* __restrict__ table, u32 li, u64 experts, u64 stride, u64 shared, u32 part, u32 base) {
    if (table) return ((const VerifyLayer*) table)[li];
    return VerifyLayer{experts, stride, shared, part, base};
}
// The plan of a layer (route_plan in route.hip.h), grid = layers, block 64 m.  The routing weights are not needed before the
// last launch and are left to a spare workgroup of launch 2 (verify_route_weights below).
extern "C" __global__ void __launch_bounds__(512) verify_plan_exl3(const float* logits, u8* plans, u32 plan_stride, u32 ioff, const u8* table, u64 shared0, u32 base, u32 ne,
                                                                   u32 k, u32 m) {
    __shared__ RoutePlanLds lds;
    const VerifyLayer L = verify_layer(table, blockIdx.x, 0, 0, shared0, 0, base);
    const u32 l = L.layer - base;
    route_plan(logits + (u64) l * m * ne, plans + (u64) l * plan_stride, ioff, ne, k, m, L.shared != 0, lds);
}

// The renormalised routing weights and the counts of the chosen experts tidx (pbuf, as the plan left it) into w and cnt:
// a wave a token, for a workgroup that has nothing else to do.
__device__ __forceinline__ void verify_route_weights(const float* __restrict__ logits, u8* __restrict__ pbuf, u32 ne, u32 k, u32 m, u32 wave, u32 lane) {
    const u32 G = m * k;
    for (u32 j = wave; j < m; j += 4) {
        u32 kk;
        const float wt = route_weights_chosen(logits + (u64) j * ne, ne, k, lane, (const u32*) pbuf + j * k, &kk);
        if (lane < k) ((float*) (pbuf + G * 4))[j * k + lane] = wt;
        if (lane == 0) ((u32*) (pbuf + 2 * G * 4))[j] = kk;
    }
}

__device__ __forceinline__ u64 uniform_u64(u64 v) {
    return ((u64) (u32) __builtin_amdgcn_readfirstlane((u32) (v >> 32)) << 32) | (u32) __builtin_amdgcn_readfirstlane((u32) v);
}

// A wave's stream of trellis rows for CT column tiles: units of UT tiles (UT / CT tile rows, 32 K UT bytes), each brought
// into one of D ring slots by NI global-to-LDS loads of 16 bytes a lane.  In LDS a unit lies packed in the order of the
// bit stream: tile row, column tile, tile word.  ONCE: past the caches, for trellises that the caches would not have at the next call either, and that push
// out what the launches share: the experts of a verify layer change with the tokens, and where the pairs are its items at most a fifth of them shares one.
// Calls with other inputs each time: layers of seven shapes at 2 to 4 bits, 1 to 8 of them alone and rounds of up to 32, 1.5 to 2 % faster whatever
// they touch, 16 MiB to 4 GiB (six of 512 experts of 2048 x 512, top-10, 4 rows, at 3 bits 250 us, 241; pairs of which 5 to 20 % repeat 1.2 %); where all
// experts together fit the last level, 256 MB, no slower.  The same inputs again and again, up to what it holds, are 0.7 % slower, at most 4.
// Projections win either way (4096 x 2048 for four inputs at 4 bits 9.2, 8.8, 6144 x 16384 at 3 bits 23.6, 22.7; 8192 x 32768, with 8 MB of partial
// sums behind it, 45.4, 46.3).  A prefill chunk's items share their expert's rows (4096 tokens 857 us, past the caches 893).
template <int K, bool H, int CT, int DEPTH = 0, int UT = 16, bool ONCE = true>
struct VerifyRing {
    static constexpr int TW = EXL3_TILE_WORDS(K, H), CH = TW / 4;   // words and 16-byte chunks a tile
    static constexpr int UR = UT / CT;                              // tile rows a unit
    static constexpr int NI = (UT * CH + 63) / 64;                  // loads a unit: UT CH chunks, 64 a load, the last load perhaps partly
    static constexpr int UW = UT * TW;                              // words a unit
    static constexpr int D = DEPTH ? DEPTH : CH <= 8 ? 3 : 2;
    u64 row0;         // the wave's first tile row, at its first column tile (uniform)
    u32 pitch;        // bytes between tile rows
    u32 units, lds;
    u32 off[NI];      // the lane's source offsets inside a unit
    __device__ __forceinline__ void init(const u8* first, u32 pitch_bytes, u32 n, u32 lds_addr, u32 lane) {
        row0 = uniform_u64((u64) first);
        pitch = pitch_bytes;
        units = n;
        lds = lds_addr;
#pragma unroll
        for (int i = 0; i < NI; i++) {
            const u32 q = 64 * i + lane, row = q / (CT * CH);
            off[i] = row * pitch + (q - row * (CT * CH)) * 16;
        }
    }
    __device__ __forceinline__ void issue(u32 unit, u32 slot, u32 lane) const {
        const u64 at = row0 + (u64) unit * ((u64) UR * pitch);
#pragma unroll
        for (int i = 0; i < NI; i++)
            if (64 * (i + 1) <= UT * CH || 64 * i + lane < (u32) (UT * CH)) lds_load_at<ONCE>(at, off[i], lds + (slot * UW + i * 256) * 4);
    }
    // requests the first D units and returns once everything requested before them has landed
    __device__ __forceinline__ void fill(u32 lane) const {
        if (units >= (u32) D) {
#pragma unroll
            for (int d = 0; d < D; d++) issue(d, d, lane);
            wait_vm<D * NI>();
        } else {
            for (u32 d = 0; d < units; d++) issue(d, d, lane);
            wait_vm<0>();
        }
    }
    // returns once at most the loads of `n` units are in flight
    __device__ __forceinline__ static void wait(u32 n) {
        switch (n) {
            case 0: wait_vm<0>(); break;
            case 1: wait_vm<NI>(); break;
            default: wait_vm<2 * NI>(); break;
        }
    }
};

// Where lane group a reads element q (0..15) of a tile row: slots 4 a .. 4 a + 3 = inputs 2 a, 2 a + 1, 2 a + 8, 2 a + 9.
__device__ __forceinline__ u32 exl3_aslot(u32 q) { return 4 * ((q & 7) >> 1) + 2 * (q >> 3) + (q & 1); }

// LDS waited for and a workgroup barrier, with no wait for the global-to-LDS loads in flight.
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// The A rows of a workgroup's 512 inputs: f16 a_sh[((step * NR + row) * 4 + a) * 8 + 4 (tile row & 1) + slot & 3], step = a
// pair of tile rows (4 a 128-block), row 3 r + part of token r, NR = 3 NMAX.  The wave holds elements `lane` and `lane + 64` of
// its 128-block kbl (0..3; 4: none) of every token's rotated inputs.  Ends with the workgroup past a barrier.
template <int NMAX>
__device__ __forceinline__ void verify_put_rows(u16* a_sh, float* s_mx, float* s_iv, const float (&rot)[NMAX][2], u32 n, u32 kbl, u32 wave, u32 lane) {
    constexpr u32 NR = 3 * NMAX;
#pragma unroll
    for (int r = 0; r < NMAX; r++) {
        if ((u32) r < n) {
            const float mx = wave_max_f32(fmaxf(__builtin_fabsf(rot[r][0]), __builtin_fabsf(rot[r][1])));
            if (lane == 0) s_mx[4 * r + wave] = mx;
        }
    }
    lds_barrier();
#pragma unroll
    for (int r = 0; r < NMAX; r++) {
        if ((u32) r < n) {
            const f32x4 mx = ((const f32x4*) s_mx)[r];
            float scale, iv;
            pow2_scale_of(f32_bits(fmaxf(fmaxf(mx[0], mx[1]), fmaxf(mx[2], mx[3]))), scale, iv);
            if (wave == 0 && lane == 0) s_iv[r] = iv;
            if (kbl < 4) {
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const u32 i = lane + 64 * h, t = i >> 4, sl = exl3_aslot(i & 15);
                    const float v = rot[r][h] * scale;
                    const _Float16 hi = (_Float16) v;
                    const float v1 = (v - (float) hi) * 0x1p11f;
                    const _Float16 mid = (_Float16) v1;
                    const _Float16 lo = (_Float16) ((v1 - (float) mid) * 0x1p11f);
                    u16* at = a_sh + (((kbl * 4 + (t >> 1)) * NR + 3 * r) * 4 + (sl >> 2)) * 8 + 4 * (t & 1) + (sl & 3);
                    at[0] = __builtin_bit_cast(u16, hi);
                    at[32] = __builtin_bit_cast(u16, mid);
                    at[64] = __builtin_bit_cast(u16, lo);
                }
            }
        }
    }
    lds_barrier();
}

// The products of one wave: its ring's units (requested up to D) against the A rows; acc[g][c]: row 4 a + part of lane group
// a = lane / 16 is part 0..2 of token 4 g + a (row 4 a + 3 belongs to nobody), column lane % 16 of column tile c.
template <int K, bool H, int CT, int NG, int NMAX>
__device__ __forceinline__ void verify_products(const VerifyRing<K, H, CT>& ring, const u32* wb, const u16* a_sh, u32 lane, f32x4 (&acc)[NG][CT]) {
    typedef VerifyRing<K, H, CT> R;
    typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
    typedef u32 u32x4v __attribute__((ext_vector_type(4)));
    constexpr bool one_shift = 16 + 3 * K + 2 * (int) H <= 32;
    constexpr u32 NR = 3 * NMAX;
    const u32 n16 = lane & 15, a = lane >> 4;
    const u32 t0 = 32 * (n16 & 7) + 8 * a + 4 * (n16 >> 3);
    // the 32 stream bits that end at bit e (exclusive) of the tile's ring: word jp holds the last of them, word jm the rest
    auto window = [&](u32 e, u32& om, u32& op, u32& sh) {
        op = (e - 1) >> 5;
        om = op == 0 ? R::TW - 1 : op - 1;
        sh = 31 - ((e - 1) & 31);
    };
    u32 om1, op1, sh1, om0 = 0, op0 = 0, sh0 = 0;
    window(H ? (t0 / 2 + 2) * (2 * K + 1) : (t0 + 4) * K, om1, op1, sh1);
    if constexpr (!one_shift) window((t0 + 2) * K, om0, op0, sh0);
    const u16* ar = a_sh + ((n16 >> 2) * 3 + min(n16 & 3, 2u)) * 32 + a * 8;
#pragma unroll
    for (int g = 0; g < NG; g++)
#pragma unroll
        for (int c = 0; c < CT; c++) acc[g][c] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    u32 slot = 0;
#pragma unroll 1
    for (u32 unit = 0; unit < ring.units; unit++) {
        R::wait(min((u32) R::D - 1, ring.units - 1 - unit));
        const u32* row = wb + slot * R::UW;
        u32 w1[16][2], w0[one_shift ? 1 : 16][2];
#pragma unroll
        for (int i = 0; i < 16; i++) {
            w1[i][0] = row[i * R::TW + om1];
            w1[i][1] = row[i * R::TW + op1];
            if constexpr (!one_shift) {
                w0[i][0] = row[i * R::TW + om0];
                w0[i][1] = row[i * R::TW + op0];
            }
        }
        u32x4v av[R::UR / 2][NG];
#pragma unroll
        for (int s = 0; s < R::UR / 2; s++)
#pragma unroll
            for (int g = 0; g < NG; g++) av[s][g] = *(const u32x4v*) (ar + ((unit * (R::UR / 2) + s) * NR + 12 * g) * 32);
        if (unit + R::D < ring.units) {
            __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0): the unit's words are in registers, its slot can take the unit D further on
            ring.issue(unit + R::D, slot, lane);
        }
        slot = slot + 1 == (u32) R::D ? 0u : slot + 1;
#pragma unroll
        for (int s = 0; s < R::UR / 2; s++) {
#pragma unroll
            for (int c = 0; c < CT; c++) {
                u32 b[2][2];
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const int i = (2 * s + h) * CT + c;
                    const u32 hi = __builtin_amdgcn_alignbit(w1[i][0], w1[i][1], sh1);
                    u32 s0, s1;
                    if constexpr (one_shift) {
                        s0 = __builtin_amdgcn_ubfe(hi, 3 * K + 2 * (int) H, 16);
                        s1 = __builtin_amdgcn_ubfe(hi, 2 * K + (int) H, 16);
                    } else {
                        const u32 lo = __builtin_amdgcn_alignbit(w0[i][0], w0[i][1], sh0);
                        s0 = __builtin_amdgcn_ubfe(lo, K, 16);
                        s1 = lo & 0xffffu;
                    }
                    const u32 s2 = __builtin_amdgcn_ubfe(hi, K + (int) H, 16), s3 = hi & 0xffffu;
                    b[h][0] = __builtin_bit_cast(u32, exl3_cb2_pair(s0, s1));
                    b[h][1] = __builtin_bit_cast(u32, exl3_cb2_pair(s2, s3));
                }
                const f16x8 bv = __builtin_bit_cast(f16x8, u32x4v{b[0][0], b[0][1], b[1][0], b[1][1]});
#pragma unroll
                for (int g = 0; g < NG; g++) acc[g][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, av[s][g]), bv, acc[g][c], 0, 0, 0);
            }
        }
    }
}

// The item's sums out of the accumulators: token 4 g + a of lane group a into out + (its pair) * stride, the wave's columns.
template <int CT, int NG>
__device__ __forceinline__ void verify_store(const f32x4 (&acc)[NG][CT], const float* s_iv, const u32 (&pairs)[4], u32 n, u64 stride, float* out, u32 lane) {
#pragma unroll
    for (int g = 0; g < NG; g++) {
        const u32 r = 4 * g + (lane >> 4);
        if (r < n) {
            const float iv = s_iv[r];
            const u64 four = (u64) pairs[2 * g] | ((u64) pairs[2 * g + 1] << 32);
            const u32 pair = (u32) (four >> (lane & 48)) & 0xffffu;
            float* o = out + (u64) pair * stride + (lane & 15);
#pragma unroll
            for (int c = 0; c < CT; c++) o[16 * c] = __builtin_fmaf(__builtin_fmaf(acc[g][c][2], 0x1p-11f, acc[g][c][1]), 0x1p-11f, acc[g][c][0]) * iv;
        }
    }
}

// One projection's products for the 512 inputs of block z and the workgroup's 64 CT columns: token r's inputs start at row(r),
// its sums go to out + (its pair) * stride + column.
template <int K, bool H, int CT, int NG, class Row>
__device__ __forceinline__ void exl3_product(const u8* bp, u32 in_f, u32 out_f, u32 z, Row row, u32 n, const u32 (&pairs)[4], u64 stride, float* __restrict__ out, u32 wave, u32 lane,
                                             u32* wb, u16* a_sh, float* s_mx, float* s_iv) {
    constexpr int NMAX = 4 * NG;
    typedef VerifyRing<K, H, CT> R;
    const u32 kbs = in_f / 128, kb = z * 4 + wave, nkb = min(4u, kbs - z * 4);
    const u32 c0 = blockIdx.x * 4 * CT + wave * CT;   // the wave's first column tile
    R ring;
    ring.init(bp + 2 * (u64) in_f + 2 * (u64) out_f + 4 + ((u64) z * 32 * (out_f / 16) + c0) * (4 * R::TW), (out_f / 16) * (4 * R::TW), nkb * 8 / R::UR,
              __builtin_amdgcn_readfirstlane(lds_offset(wb)), lane);
    // the wave's 128-block of every token and its scales, then the first units of its rows behind them, uncounted.  Every load
    // is made, past the item's tokens and blocks of an earlier one: a load behind a branch would leave its register to be
    // copied at the branches' end, before the value is there.
    float v[NMAX][2];
    const u32 kbc = min(kb, kbs - 1);
    const u16* suh = (const u16*) bp + kbc * 128;
    u32 sc0 = load_u16_uncounted(suh + lane), sc1 = load_u16_uncounted(suh + lane + 64);
#pragma unroll
    for (int r = 0; r < NMAX; r++) {
        const float* xj = row(min((u32) r, n - 1)) + kbc * 128;
        v[r][0] = load_f32_uncounted(xj + lane);
        v[r][1] = load_f32_uncounted(xj + lane + 64);
    }
    ring.fill(lane);
    load_landed(sc0);
    load_landed(sc1);
#pragma unroll
    for (int r = 0; r < NMAX; r++) {
        load_landed(v[r][0]);
        load_landed(v[r][1]);
    }
#pragma unroll
    for (int r = 0; r < NMAX; r++) {
        if ((u32) r < n) {
            v[r][0] *= f16_to_f32((u16) sc0);
            v[r][1] *= f16_to_f32((u16) sc1);
            wht128_wave(v[r][0], v[r][1], lane);
            if (kb >= kbs) v[r][0] = v[r][1] = 0.0f;
        }
    }
    verify_put_rows<NMAX>(a_sh, s_mx, s_iv, v, n, kb < kbs ? wave : 4u, wave, lane);
    f32x4 acc[NG][CT];
    verify_products<K, H, CT, NG, NMAX>(ring, wb, a_sh, lane, acc);
    verify_store<CT, NG>(acc, s_iv, pairs, n, stride, out + c0 * 16, lane);
}

// The shared expert's item: every token, pairs m k + j.
__device__ __forceinline__ void verify_shared_item(u32 G, u64& toks, u32 (&pairs)[4]) {
    toks = 0x0706050403020100ull;
#pragma unroll
    for (int i = 0; i < 4; i++) pairs[i] = (G + 2 * i) | ((G + 2 * i + 1) << 16);
}

// Launch 2: the gate and up products of every item, gup[(((layer * 2 + sel) * S + pair) * zs + z) * ff + column], S = m (k + 1),
// sel 0 = gate, 1 = up, z = the block of 512 inputs.  grid = (ff / (64 CT), 2 slots, layers zs), slots = m k + 2: at least one
// more than a layer can have items.  block 256.
// ioff = 0 (one layer): there is no plan, launch 1 does not run.  The items are the shared expert and then the (token,
// rank) pairs, one token each (slots = m k + 1); the workgroups select for themselves and launch 3 works the weights out.  A layer of a
// call of its own takes this form where few tokens can share an expert: the pairs' weights are decoded once each, which
// costs less than another launch ahead of everything.  A token's sums do not depend on the other tokens of an item: both
// forms give the same bits.
template <int K, bool H, int CT, int NG>
__device__ __forceinline__ void verify_gate_up_kernel(const float* __restrict__ logits, const u8* __restrict__ table, u64 experts, u64 stride, u64 shared, u32 part,
                                                      u32 base, const u8* __restrict__ plans, u8* __restrict__ weights, u32 plan_stride, u32 ioff, const float* __restrict__ u, float* __restrict__ gup, u32 ne, u32 k, u32 m,
                                                      u32 hidden, u32 ff) {
    constexpr int NMAX = 4 * NG;
    typedef VerifyRing<K, H, CT> R;
    __shared__ __attribute__((aligned(16))) u32 wb_all[4][R::D * R::UW];
    __shared__ __attribute__((aligned(16))) u16 a_sh[16 * 3 * NMAX * 32];
    __shared__ __attribute__((aligned(16))) float s_mx[4 * NMAX];
    __shared__ float s_iv[NMAX];
    __shared__ u32 s_top[16];
    static_assert(sizeof(a_sh) >= 512 * sizeof(double), "the exact selection's scratch");
    const u32 wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const u32 zs = (hidden / 128 + 3) / 4, li = blockIdx.z / zs, z = blockIdx.z - li * zs;
    const u32 slots = gridDim.y >> 1, sel = blockIdx.y >= slots ? 1u : 0u, it = blockIdx.y - sel * slots;
    const VerifyLayer L = verify_layer(table, li, experts, stride, shared, part, base);
    const u32 l = L.layer - base;
    const u32 G = m * k, S = G + m;
    u32 e, n, pairs[4];
    u64 toks;
    if (ioff) {
        const u32* plan = (const u32*) (plans + (u64) l * plan_stride + ioff);
        const u32* rec = plan + 4 + 8 * it;   // there for every slot, an item or not: read along with the count
        e = rec[0];
        n = __builtin_amdgcn_readfirstlane(min(rec[1], (u32) NMAX));
        toks = (u64) rec[2] | ((u64) rec[3] << 32);
#pragma unroll
        for (int i = 0; i < 4; i++) pairs[i] = __builtin_amdgcn_readfirstlane(rec[4 + i]);
        if (it >= plan[0]) {
            // the last slot is never an item: one of its workgroups works the layer's routing weights out for the last launch
            // while the others multiply
            if (blockIdx.y == gridDim.y - 1 && blockIdx.x == 0 && z == 0)
                verify_route_weights(logits + (u64) l * m * ne, weights + (u64) l * plan_stride, ne, k, m, wave, lane);
            return;
        }
    } else if (it > 0) {
        // no plan: a workgroup redoes its token's selection on one of its waves (not always the same one: the prologues of
        // co-resident workgroups spread over the SIMDs), ahead of the decoding waves of other workgroups on its SIMD
        const u32 pair = it - 1, j = pair / k, t = pair - j * k;
        if (wave == (blockIdx.x + blockIdx.y + blockIdx.z) % 4) {
            __builtin_amdgcn_s_setprio(3);
            route_id_of_rank(logits + (u64) j * ne, ne, k, t, lane, (double*) &a_sh[0], s_top);   // only s_top[t] is read
            __builtin_amdgcn_s_setprio(0);
            if (sel == 0 && blockIdx.x == 0 && z == 0 && lane == 0) ((u32*) weights)[pair] = s_top[t];
        }
        __syncthreads();
        e = __builtin_amdgcn_readfirstlane(s_top[t]);
        if (e == 0xffffffffu) return;
        n = 1;
        toks = j;
        pairs[0] = pair;
        pairs[1] = pairs[2] = pairs[3] = 0;
    } else {
        if (!L.shared) return;
        e = 0xffffffffu;
        n = m;
        verify_shared_item(G, toks, pairs);
    }
    const u8* bp = (const u8*) uniform_u64((e == 0xffffffffu ? L.shared : L.experts + e * L.stride) + (u64) sel * L.part);
    exl3_product<K, H, CT, NG>(bp, hidden, ff, z, [&](u32 r) { return u + ((u64) l * m + ((u32) (toks >> (8 * r)) & 0xffu)) * hidden; }, n, pairs, (u64) zs * ff,
                               gup + (((u64) (li * 2 + sel) * S) * zs + z) * ff, wave, lane, wb_all[wave], a_sh, s_mx, s_iv);
}

// Launch 3: act = silu(gate) * up of every token of the item out of launch 2's sums (partials added, output side of the two
// projections), rotated into the down projection's basis as A rows, then its products: dn[((layer * S + pair) * zd + z) *
// hidden + column], zd = ceil(ff / 512).  grid = (hidden / (64 CT), slots, layers zd), block 256.  WIDE: gate and up have more than four
// partials (inputs of more than 2048 features), which are asked for eight at once (four layers of 32 experts of 4096 x 1536, top-2, 8 rows, at 4 bits 350 us, 324;
// of 64 of 4096 x 512, top-4, 2 rows 120.5, 116.5; six of 160 of 3584 x 768, top-12, 6 rows, at 3 bits 725, 712).  Kernels of their own: as a
// branch, 10 KB of code more, the others lose (a round of 16 layers of 1024 x 768 at 8 rows 232 us, 237).
template <int K, bool H, int CT, int NG, bool WIDE = false>
__device__ __forceinline__ void verify_down_kernel(const float* __restrict__ logits, const u8* __restrict__ table, u64 experts, u64 stride, u64 shared, u32 part0, u32 base,
                                                   const u8* __restrict__ plans, u8* __restrict__ weights, u32 plan_stride, u32 ioff, const float* __restrict__ gup, float* __restrict__ dn,
                                                   u32 ne, u32 k, u32 m, u32 hidden, u32 ff) {
    constexpr int NMAX = 4 * NG, TOKENS = WIDE ? 1 : 2, PARTS = WIDE ? 8 : 4;
    typedef VerifyRing<K, H, CT> R;
    __shared__ __attribute__((aligned(16))) u32 wb_all[4][R::D * R::UW];
    __shared__ __attribute__((aligned(16))) u16 a_sh[16 * 3 * NMAX * 32];
    __shared__ __attribute__((aligned(16))) float s_mx[4 * NMAX];
    __shared__ float s_iv[NMAX];
    const u32 wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const u32 zs = (hidden / 128 + 3) / 4, zd = (ff / 128 + 3) / 4, li = blockIdx.z / zd, z = blockIdx.z - li * zd, it = blockIdx.y;
    const VerifyLayer L = verify_layer(table, li, experts, stride, shared, part0, base);
    const u8* pbuf = plans + (u64) (L.layer - base) * plan_stride;
    const u32 G = m * k, S = G + m;
    u32 e, n, pairs[4];
    if (ioff) {
        const u32* plan = (const u32*) (pbuf + ioff);
        const u32* rec = plan + 4 + 8 * it;
        e = rec[0];
        n = __builtin_amdgcn_readfirstlane(min(rec[1], (u32) NMAX));
#pragma unroll
        for (int i = 0; i < 4; i++) pairs[i] = __builtin_amdgcn_readfirstlane(rec[4 + i]);
        if (it >= plan[0]) return;
    } else if (it > 0) {
        const u32 pair = it - 1;
        if (pair % k == 0 && blockIdx.x == 0 && z == 0 && wave == 3) {
            // one wave a token: the routing weights and the count, for launch 4 (nothing in this launch reads them)
            const u32 j = pair / k;
            u32 kk;
            const float wt = route_weights_chosen(logits + (u64) j * ne, ne, k, lane, (const u32*) pbuf + pair, &kk);
            if (lane < k) ((float*) (weights + G * 4))[pair + lane] = wt;
            if (lane == 0) ((u32*) (weights + 2 * G * 4))[j] = kk;
        }
        e = ((const u32*) pbuf)[pair];
        if (e == 0xffffffffu) return;
        n = 1;
        pairs[0] = pair;
        pairs[1] = pairs[2] = pairs[3] = 0;
    } else {
        if (!L.shared) return;
        u64 toks;
        e = 0xffffffffu;
        n = m;
        verify_shared_item(G, toks, pairs);
    }
    const u8* bp = (const u8*) uniform_u64(e == 0xffffffffu ? L.shared : L.experts + e * L.stride);
    const u64 part = L.part;
    const u32 kbs = ff / 128, kb = z * 4 + wave, nkb = min(4u, kbs - z * 4);
    float rot[NMAX][2];
#pragma unroll
    for (int r = 0; r < NMAX; r++) rot[r][0] = rot[r][1] = 0.0f;
    const u32 c0 = blockIdx.x * 4 * CT + wave * CT;
    R ring;
    ring.init(bp + 2 * part + 2 * (u64) ff + 2 * (u64) hidden + 4 + ((u64) z * 32 * (hidden / 16) + c0) * (4 * R::TW), (hidden / 16) * (4 * R::TW),
              nkb * 8 / R::UR, __builtin_amdgcn_readfirstlane(lds_offset(wb_all[wave])), lane);
    if (kb < kbs) {
        const float* g0 = gup + ((u64) li * 2 * S * zs) * ff + kb * 128 + lane;
        // gate's and up's output scales and down's input scales of the block
        u32 sc[6];
        const u16* svg = (const u16*) (bp + 2 * (u64) hidden) + kb * 128 + lane;
        const u16* svu = (const u16*) (bp + part + 2 * (u64) hidden) + kb * 128 + lane;
        const u16* sud = (const u16*) (bp + 2 * part) + kb * 128 + lane;
        sc[0] = load_u16_uncounted(svg);
        sc[1] = load_u16_uncounted(svg + 64);
        sc[2] = load_u16_uncounted(svu);
        sc[3] = load_u16_uncounted(svu + 64);
        sc[4] = load_u16_uncounted(sud);
        sc[5] = load_u16_uncounted(sud + 64);
#pragma unroll
        for (int r0 = 0; r0 < NMAX; r0 += TOKENS) {
            if ((u32) r0 < n) {
                // two tokens at a time, the first four partials of each requested together (WIDE: one, its first eight); the first lot goes out
                // ahead of the rows
                float pv[TOKENS][PARTS][4];
#pragma unroll
                for (int q = 0; q < TOKENS; q++) {
                    // (a lot's second token past the item's: its first again, so that no load stands behind a branch)
                    const u32 pair = ((u32) (r0 + q) < n ? pairs[r0 / 2] >> (16 * ((r0 + q) & 1)) : pairs[r0 / 2]) & 0xffffu;
                    const float* pg = g0 + (u64) pair * zs * ff;
                    const float* pu = g0 + (u64) (S + pair) * zs * ff;
#pragma unroll
                    for (int zz = 0; zz < PARTS; zz++) {
                        const u64 o = (u64) min((u32) zz, zs - 1) * ff;
                        pv[q][zz][0] = load_f32_uncounted(pg + o);
                        pv[q][zz][1] = load_f32_uncounted(pg + o + 64);
                        pv[q][zz][2] = load_f32_uncounted(pu + o);
                        pv[q][zz][3] = load_f32_uncounted(pu + o + 64);
                    }
                }
                if (r0 == 0) {
                    ring.fill(lane);
#pragma unroll
                    for (int i = 0; i < 6; i++) load_landed(sc[i]);
                } else {
                    wait_vm<0>();
                }
#pragma unroll
                for (int q = 0; q < TOKENS; q++)
#pragma unroll
                    for (int zz = 0; zz < PARTS; zz++)
#pragma unroll
                        for (int c = 0; c < 4; c++) load_landed(pv[q][zz][c]);
#pragma unroll
                for (int q = 0; q < TOKENS; q++) {
                    const int r = r0 + q;
                    if ((u32) r < n) {
                        float t[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                        for (int zz = 0; zz < PARTS; zz++)
#pragma unroll
                            for (int c = 0; c < 4; c++) t[c] += (u32) zz < zs ? pv[q][zz][c] : 0.0f;
                        if (zs > (u32) PARTS) {
                            const u32 pair = (pairs[r / 2] >> (16 * (r & 1))) & 0xffffu;
                            for (u32 zz = PARTS; zz < zs; zz++) {
                                const float* pg = g0 + ((u64) pair * zs + zz) * ff;
                                const float* pu = g0 + ((u64) (S + pair) * zs + zz) * ff;
                                t[0] += pg[0];
                                t[1] += pg[64];
                                t[2] += pu[0];
                                t[3] += pu[64];
                            }
                        }
                        wht128_wave(t[0], t[1], lane);
                        wht128_wave(t[2], t[3], lane);
                        rot[r][0] = siluf_ref(t[0] * f16_to_f32((u16) sc[0])) * (t[2] * f16_to_f32((u16) sc[2])) * f16_to_f32((u16) sc[4]);
                        rot[r][1] = siluf_ref(t[1] * f16_to_f32((u16) sc[1])) * (t[3] * f16_to_f32((u16) sc[3])) * f16_to_f32((u16) sc[5]);
                        wht128_wave(rot[r][0], rot[r][1], lane);
                    }
                }
            }
        }
    } else {
        ring.fill(lane);
    }
    verify_put_rows<NMAX>(a_sh, s_mx, s_iv, rot, n, kb < kbs ? wave : 4u, wave, lane);
    f32x4 acc[NG][CT];
    verify_products<K, H, CT, NG, NMAX>(ring, wb_all[wave], a_sh, lane, acc);
    verify_store<CT, NG>(acc, s_iv, pairs, n, (u64) zd * hidden, dn + ((u64) li * S * zd + z) * hidden + c0 * 16, lane);
}

// Occupancy: workgroups a compute unit's LDS (160 KiB) holds; the register budget follows it.
#define EXL3_VERIFY_OCC(K, NG) ((NG) == 1 ? ((K) <= 2 ? 6 : (K) == 3 ? 5 : (K) <= 6 ? 4 : 3) : ((K) <= 2 ? 4 : 3))
// CT = 8 column tiles a wave (plain name), or 4 or 2 (t4, t2: shorter waves, for launches that would leave the chip idle);
// w: batches of more than 4 rows.
#define EXL3_VERIFY_ENTRIES(K) \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K, 1)) verify_gate_up_exl3_##K(const float* logits, const u8* table, u64 experts, u64 stride, u64 shared, u32 part, u32 base, \
        const u8* plans, u8* weights, u32 plan_stride, u32 ioff, const float* u, float* gup, u32 ne, u32 k, u32 m, u32 hidden, u32 ff) { \
        verify_gate_up_kernel<K, false, 8, 1>(logits, table, experts, stride, shared, part, base, plans, weights, plan_stride, ioff, u, gup, ne, k, m, hidden, ff); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K, 1)) verify_down_exl3_##K(const float* logits, const u8* table, u64 experts, u64 stride, u64 shared, u32 part, u32 base, \
        const u8* plans, u8* weights, u32 plan_stride, u32 ioff, const float* gup, float* dn, u32 ne, u32 k, u32 m, u32 hidden, u32 ff) { \
        verify_down_kernel<K, false, 8, 1>(logits, table, experts, stride, shared, part, base, plans, weights, plan_stride, ioff, gup, dn, ne, k, m, hidden, ff); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K, 1)) verify_gate_up_t4_exl3_##K(const float* logits, const u8* table, u64 experts, u64 stride, u64 shared, u32 part, u32 base, \
        const u8* plans, u8* weights, u32 plan_stride, u32 ioff, const float* u, float* gup, u32 ne, u32 k, u32 m, u32 hidden, u32 ff) { \
        verify_gate_up_kernel<K, false, 4, 1>(logits, table, experts, stride, shared, part, base, plans, weights, plan_stride, ioff, u, gup, ne, k, m, hidden, ff); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K, 1)) verify_down_t4_exl3_##K(const float* logits, const u8* table, u64 experts, u64 stride, u64 shared, u32 part, u32 base, \
        const u8* plans, u8* weights, u32 plan_stride, u32 ioff, const float* gup, float* dn, u32 ne, u32 k, u32 m, u32 hidden, u32 ff) { \
        verify_down_kernel<K, false, 4, 1>(logits, table, experts, stride, shared, part, base, plans, weights, plan_stride, ioff, gup, dn, ne, k, m, hidden, ff); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K, 1)) verify_gate_up_t2_exl3_##K(const float* logits, const u8* table, u64 experts, u64 stride, u64 shared, u32 part, u32 base, \
        const u8* plans, u8* weights, u32 plan_stride, u32 ioff, const float* u, float* gup, u32 ne, u32 k, u32 m, u32 hidden, u32 ff) { \
        verify_gate_up_kernel<K, false, 2, 1>(logits, table, experts, stride, shared, part, base, plans, weights, plan_stride, ioff, u, gup, ne, k, m, hidden, ff); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K, 1)) verify_down_t2_exl3_##K(const float* logits, const u8* table, u64 experts, u64 stride, u64 shared, u32 part, u32 base, \
        const u8* plans, u8* weights, u32 plan_stride, u32 ioff, const float* gup, float* dn, u32 ne, u32 k, u32 m, u32 hidden, u32 ff) { \
        verify_down_kernel<K, false, 2, 1>(logits, table, experts, stride, shared, part, base, plans, weights, plan_stride, ioff, gup, dn, ne, k, m, hidden, ff); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K, 2)) verify_gate_up_w_exl3_##K(const float* logits, const u8* table, u64 experts, u64 stride, u64 shared, u32 part, u32 base, \
        const u8* plans, u8* weights, u32 plan_stride, u32 ioff, const float* u, float* gup, u32 ne, u32 k, u32 m, u32 hidden, u32 ff) { \
        verify_gate_up_kernel<K, false, 8, 2>(logits, table, experts, stride, shared, part, base, plans, weights, plan_stride, ioff, u, gup, ne, k, m, hidden, ff); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K, 2)) verify_down_w_exl3_##K(const float* logits, const u8* table, u64 experts, u64 stride, u64 shared, u32 part, u32 base, \
        const u8* plans, u8* weights, u32 plan_stride, u32 ioff, const float* gup, float* dn, u32 ne, u32 k, u32 m, u32 hidden, u32 ff) { \
        verify_down_kernel<K, false, 8, 2>(logits, table, experts, stride, shared, part, base, plans, weights, plan_stride, ioff, gup, dn, ne, k, m, hidden, ff); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K, 2)) verify_gate_up_t4w_exl3_##K(const float* logits, const u8* table, u64 experts, u64 stride, u64 shared, u32 part, u32 base, \
        const u8* plans, u8* weights, u32 plan_stride, u32 ioff, const float* u, float* gup, u32 ne, u32 k, u32 m, u32 hidden, u32 ff) { \
        verify_gate_up_kernel<K, false, 4, 2>(logits, table, experts, stride, shared, part, base, plans, weights, plan_stride, ioff, u, gup, ne, k, m, hidden, ff); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K, 2)) verify_down_t4w_exl3_##K(const float* logits, const u8* table, u64 experts, u64 stride, u64 shared, u32 part, u32 base, \
        const u8* plans, u8* weights, u32 plan_stride, u32 ioff, const float* gup, float* dn, u32 ne, u32 k, u32 m, u32 hidden, u32 ff) { \
        verify_down_kernel<K, false, 4, 2>(logits, table, experts, stride, shared, part, base, plans, weights, plan_stride, ioff, gup, dn, ne, k, m, hidden, ff); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K, 2)) verify_gate_up_t2w_exl3_##K(const float* logits, const u8* table, u64 experts, u64 stride, u64 shared, u32 part, u32 base, \
        const u8* plans, u8* weights, u32 plan_stride, u32 ioff, const float* u, float* gup, u32 ne, u32 k, u32 m, u32 hidden, u32 ff) { \
        verify_gate_up_kernel<K, false, 2, 2>(logits, table, experts, stride, shared, part, base, plans, weights, plan_stride, ioff, u, gup, ne, k, m, hidden, ff); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K, 2)) verify_down_t2w_exl3_##K(const float* logits, const u8* table, u64 experts, u64 stride, u64 shared, u32 part, u32 base, \
        const u8* plans, u8* weights, u32 plan_stride, u32 ioff, const float* gup, float* dn, u32 ne, u32 k, u32 m, u32 hidden, u32 ff) { \
        verify_down_kernel<K, false, 2, 2>(logits, table, experts, stride, shared, part, base, plans, weights, plan_stride, ioff, gup, dn, ne, k, m, hidden, ff); \
    }
#define EXL3_VERIFY_HALF_ENTRIES(K) \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K + 1, 1)) verify_gate_up_exl3h_##K(const float* logits, const u8* table, u64 experts, u64 stride, u64 shared, u32 part, u32 base, \
        const u8* plans, u8* weights, u32 plan_stride, u32 ioff, const float* u, float* gup, u32 ne, u32 k, u32 m, u32 hidden, u32 ff) { \
        verify_gate_up_kernel<K, true, 8, 1>(logits, table, experts, stride, shared, part, base, plans, weights, plan_stride, ioff, u, gup, ne, k, m, hidden, ff); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K + 1, 1)) verify_down_exl3h_##K(const float* logits, const u8* table, u64 experts, u64 stride, u64 shared, u32 part, u32 base, \
        const u8* plans, u8* weights, u32 plan_stride, u32 ioff, const float* gup, float* dn, u32 ne, u32 k, u32 m, u32 hidden, u32 ff) { \
        verify_down_kernel<K, true, 8, 1>(logits, table, experts, stride, shared, part, base, plans, weights, plan_stride, ioff, gup, dn, ne, k, m, hidden, ff); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K + 1, 1)) verify_gate_up_t4_exl3h_##K(const float* logits, const u8* table, u64 experts, u64 stride, u64 shared, u32 part, u32 base, \
        const u8* plans, u8* weights, u32 plan_stride, u32 ioff, const float* u, float* gup, u32 ne, u32 k, u32 m, u32 hidden, u32 ff) { \
        verify_gate_up_kernel<K, true, 4, 1>(logits, table, experts, stride, shared, part, base, plans, weights, plan_stride, ioff, u, gup, ne, k, m, hidden, ff); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K + 1, 1)) verify_down_t4_exl3h_##K(const float* logits, const u8* table, u64 experts, u64 stride, u64 shared, u32 part, u32 base, \
        const u8* plans, u8* weights, u32 plan_stride, u32 ioff, const float* gup, float* dn, u32 ne, u32 k, u32 m, u32 hidden, u32 ff) { \
        verify_down_kernel<K, true, 4, 1>(logits, table, experts, stride, shared, part, base, plans, weights, plan_stride, ioff, gup, dn, ne, k, m, hidden, ff); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K + 1, 1)) verify_gate_up_t2_exl3h_##K(const float* logits, const u8* table, u64 experts, u64 stride, u64 shared, u32 part, u32 base, \
        const u8* plans, u8* weights, u32 plan_stride, u32 ioff, const float* u, float* gup, u32 ne, u32 k, u32 m, u32 hidden, u32 ff) { \
        verify_gate_up_kernel<K, true, 2, 1>(logits, table, experts, stride, shared, part, base, plans, weights, plan_stride, ioff, u, gup, ne, k, m, hidden, ff); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K + 1, 1)) verify_down_t2_exl3h_##K(const float* logits, const u8* table, u64 experts, u64 stride, u64 shared, u32 part, u32 base, \
        const u8* plans, u8* weights, u32 plan_stride, u32 ioff, const float* gup, float* dn, u32 ne, u32 k, u32 m, u32 hidden, u32 ff) { \
        verify_down_kernel<K, true, 2, 1>(logits, table, experts, stride, shared, part, base, plans, weights, plan_stride, ioff, gup, dn, ne, k, m, hidden, ff); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K + 1, 2)) verify_gate_up_w_exl3h_##K(const float* logits, const u8* table, u64 experts, u64 stride, u64 shared, u32 part, u32 base, \
        const u8* plans, u8* weights, u32 plan_stride, u32 ioff, const float* u, float* gup, u32 ne, u32 k, u32 m, u32 hidden, u32 ff) { \
        verify_gate_up_kernel<K, true, 8, 2>(logits, table, experts, stride, shared, part, base, plans, weights, plan_stride, ioff, u, gup, ne, k, m, hidden, ff); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K + 1, 2)) verify_down_w_exl3h_##K(const float* logits, const u8* table, u64 experts, u64 stride, u64 shared, u32 part, u32 base, \
        const u8* plans, u8* weights, u32 plan_stride, u32 ioff, const float* gup, float* dn, u32 ne, u32 k, u32 m, u32 hidden, u32 ff) { \
        verify_down_kernel<K, true, 8, 2>(logits, table, experts, stride, shared, part, base, plans, weights, plan_stride, ioff, gup, dn, ne, k, m, hidden, ff); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K + 1, 2)) verify_gate_up_t4w_exl3h_##K(const float* logits, const u8* table, u64 experts, u64 stride, u64 shared, u32 part, u32 base, \
        const u8* plans, u8* weights, u32 plan_stride, u32 ioff, const float* u, float* gup, u32 ne, u32 k, u32 m, u32 hidden, u32 ff) { \
        verify_gate_up_kernel<K, true, 4, 2>(logits, table, experts, stride, shared, part, base, plans, weights, plan_stride, ioff, u, gup, ne, k, m, hidden, ff); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K + 1, 2)) verify_down_t4w_exl3h_##K(const float* logits, const u8* table, u64 experts, u64 stride, u64 shared, u32 part, u32 base, \
        const u8* plans, u8* weights, u32 plan_stride, u32 ioff, const float* gup, float* dn, u32 ne, u32 k, u32 m, u32 hidden, u32 ff) { \
        verify_down_kernel<K, true, 4, 2>(logits, table, experts, stride, shared, part, base, plans, weights, plan_stride, ioff, gup, dn, ne, k, m, hidden, ff); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K + 1, 2)) verify_gate_up_t2w_exl3h_##K(const float* logits, const u8* table, u64 experts, u64 stride, u64 shared, u32 part, u32 base, \
        const u8* plans, u8* weights, u32 plan_stride, u32 ioff, const float* u, float* gup, u32 ne, u32 k, u32 m, u32 hidden, u32 ff) { \
        verify_gate_up_kernel<K, true, 2, 2>(logits, table, experts, stride, shared, part, base, plans, weights, plan_stride, ioff, u, gup, ne, k, m, hidden, ff); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K + 1, 2)) verify_down_t2w_exl3h_##K(const float* logits, const u8* table, u64 experts, u64 stride, u64 shared, u32 part, u32 base, \
        const u8* plans, u8* weights, u32 plan_stride, u32 ioff, const float* gup, float* dn, u32 ne, u32 k, u32 m, u32 hidden, u32 ff) { \
        verify_down_kernel<K, true, 2, 2>(logits, table, experts, stride, shared, part, base, plans, weights, plan_stride, ioff, gup, dn, ne, k, m, hidden, ff); \
    }
// x: inputs of more than 2048 features
#define EXL3_VERIFY_WIDE_ENTRIES(K) \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K, 1)) verify_down_x_exl3_##K(const float* logits, const u8* table, u64 experts, u64 stride, u64 shared, u32 part, u32 base, \
        const u8* plans, u8* weights, u32 plan_stride, u32 ioff, const float* gup, float* dn, u32 ne, u32 k, u32 m, u32 hidden, u32 ff) { \
        verify_down_kernel<K, false, 8, 1, true>(logits, table, experts, stride, shared, part, base, plans, weights, plan_stride, ioff, gup, dn, ne, k, m, hidden, ff); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K, 1)) verify_down_x_t4_exl3_##K(const float* logits, const u8* table, u64 experts, u64 stride, u64 shared, u32 part, u32 base, \
        const u8* plans, u8* weights, u32 plan_stride, u32 ioff, const float* gup, float* dn, u32 ne, u32 k, u32 m, u32 hidden, u32 ff) { \
        verify_down_kernel<K, false, 4, 1, true>(logits, table, experts, stride, shared, part, base, plans, weights, plan_stride, ioff, gup, dn, ne, k, m, hidden, ff); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K, 1)) verify_down_x_t2_exl3_##K(const float* logits, const u8* table, u64 experts, u64 stride, u64 shared, u32 part, u32 base, \
        const u8* plans, u8* weights, u32 plan_stride, u32 ioff, const float* gup, float* dn, u32 ne, u32 k, u32 m, u32 hidden, u32 ff) { \
        verify_down_kernel<K, false, 2, 1, true>(logits, table, experts, stride, shared, part, base, plans, weights, plan_stride, ioff, gup, dn, ne, k, m, hidden, ff); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K, 2)) verify_down_x_w_exl3_##K(const float* logits, const u8* table, u64 experts, u64 stride, u64 shared, u32 part, u32 base, \
        const u8* plans, u8* weights, u32 plan_stride, u32 ioff, const float* gup, float* dn, u32 ne, u32 k, u32 m, u32 hidden, u32 ff) { \
        verify_down_kernel<K, false, 8, 2, true>(logits, table, experts, stride, shared, part, base, plans, weights, plan_stride, ioff, gup, dn, ne, k, m, hidden, ff); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K, 2)) verify_down_x_t4w_exl3_##K(const float* logits, const u8* table, u64 experts, u64 stride, u64 shared, u32 part, u32 base, \
        const u8* plans, u8* weights, u32 plan_stride, u32 ioff, const float* gup, float* dn, u32 ne, u32 k, u32 m, u32 hidden, u32 ff) { \
        verify_down_kernel<K, false, 4, 2, true>(logits, table, experts, stride, shared, part, base, plans, weights, plan_stride, ioff, gup, dn, ne, k, m, hidden, ff); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K, 2)) verify_down_x_t2w_exl3_##K(const float* logits, const u8* table, u64 experts, u64 stride, u64 shared, u32 part, u32 base, \
        const u8* plans, u8* weights, u32 plan_stride, u32 ioff, const float* gup, float* dn, u32 ne, u32 k, u32 m, u32 hidden, u32 ff) { \
        verify_down_kernel<K, false, 2, 2, true>(logits, table, experts, stride, shared, part, base, plans, weights, plan_stride, ioff, gup, dn, ne, k, m, hidden, ff); \
    }
#define EXL3_VERIFY_WIDE_HALF_ENTRIES(K) \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K + 1, 1)) verify_down_x_exl3h_##K(const float* logits, const u8* table, u64 experts, u64 stride, u64 shared, u32 part, u32 base, \
        const u8* plans, u8* weights, u32 plan_stride, u32 ioff, const float* gup, float* dn, u32 ne, u32 k, u32 m, u32 hidden, u32 ff) { \
        verify_down_kernel<K, true, 8, 1, true>(logits, table, experts, stride, shared, part, base, plans, weights, plan_stride, ioff, gup, dn, ne, k, m, hidden, ff); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K + 1, 1)) verify_down_x_t4_exl3h_##K(const float* logits, const u8* table, u64 experts, u64 stride, u64 shared, u32 part, u32 base, \
        const u8* plans, u8* weights, u32 plan_stride, u32 ioff, const float* gup, float* dn, u32 ne, u32 k, u32 m, u32 hidden, u32 ff) { \
        verify_down_kernel<K, true, 4, 1, true>(logits, table, experts, stride, shared, part, base, plans, weights, plan_stride, ioff, gup, dn, ne, k, m, hidden, ff); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K + 1, 1)) verify_down_x_t2_exl3h_##K(const float* logits, const u8* table, u64 experts, u64 stride, u64 shared, u32 part, u32 base, \
        const u8* plans, u8* weights, u32 plan_stride, u32 ioff, const float* gup, float* dn, u32 ne, u32 k, u32 m, u32 hidden, u32 ff) { \
        verify_down_kernel<K, true, 2, 1, true>(logits, table, experts, stride, shared, part, base, plans, weights, plan_stride, ioff, gup, dn, ne, k, m, hidden, ff); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K + 1, 2)) verify_down_x_w_exl3h_##K(const float* logits, const u8* table, u64 experts, u64 stride, u64 shared, u32 part, u32 base, \
        const u8* plans, u8* weights, u32 plan_stride, u32 ioff, const float* gup, float* dn, u32 ne, u32 k, u32 m, u32 hidden, u32 ff) { \
        verify_down_kernel<K, true, 8, 2, true>(logits, table, experts, stride, shared, part, base, plans, weights, plan_stride, ioff, gup, dn, ne, k, m, hidden, ff); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K + 1, 2)) verify_down_x_t4w_exl3h_##K(const float* logits, const u8* table, u64 experts, u64 stride, u64 shared, u32 part, u32 base, \
        const u8* plans, u8* weights, u32 plan_stride, u32 ioff, const float* gup, float* dn, u32 ne, u32 k, u32 m, u32 hidden, u32 ff) { \
        verify_down_kernel<K, true, 4, 2, true>(logits, table, experts, stride, shared, part, base, plans, weights, plan_stride, ioff, gup, dn, ne, k, m, hidden, ff); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K + 1, 2)) verify_down_x_t2w_exl3h_##K(const float* logits, const u8* table, u64 experts, u64 stride, u64 shared, u32 part, u32 base, \
        const u8* plans, u8* weights, u32 plan_stride, u32 ioff, const float* gup, float* dn, u32 ne, u32 k, u32 m, u32 hidden, u32 ff) { \
        verify_down_kernel<K, true, 2, 2, true>(logits, table, experts, stride, shared, part, base, plans, weights, plan_stride, ioff, gup, dn, ne, k, m, hidden, ff); \
    }
EXL3_VERIFY_ENTRIES(1)
EXL3_VERIFY_ENTRIES(2)
EXL3_VERIFY_ENTRIES(3)
EXL3_VERIFY_ENTRIES(4)
EXL3_VERIFY_ENTRIES(5)
EXL3_VERIFY_ENTRIES(6)
EXL3_VERIFY_ENTRIES(7)
EXL3_VERIFY_ENTRIES(8)
EXL3_VERIFY_HALF_ENTRIES(1)
EXL3_VERIFY_HALF_ENTRIES(2)
EXL3_VERIFY_HALF_ENTRIES(3)
EXL3_VERIFY_WIDE_ENTRIES(1)
EXL3_VERIFY_WIDE_ENTRIES(2)
EXL3_VERIFY_WIDE_ENTRIES(3)
EXL3_VERIFY_WIDE_ENTRIES(4)
EXL3_VERIFY_WIDE_ENTRIES(5)
EXL3_VERIFY_WIDE_ENTRIES(6)
EXL3_VERIFY_WIDE_ENTRIES(7)
EXL3_VERIFY_WIDE_ENTRIES(8)
EXL3_VERIFY_WIDE_HALF_ENTRIES(1)
EXL3_VERIFY_WIDE_HALF_ENTRIES(2)
EXL3_VERIFY_WIDE_HALF_ENTRIES(3)

// Launch 4: token j = blockIdx.y of layer blockIdx.z, output block blockIdx.x: y[j] = sum over its cnt[j] experts t, in rank order,
// of w[j,t] * (the down product of pair j k + t) + sigmoid(gl[j]) * (the shared expert's).  Wave t finishes expert t (partials
// added, output-side transform, scales; the shared one on a wave of its own, or on wave 0 at k = 16), then the first two waves
// add them up in rank order (moe_combine_qwen_rows, kernels/forward.cu:2568).  grid = (hidden / 128, m, layers), block 64 times
// the experts of a token (at most 1024).
extern "C" __global__ void __launch_bounds__(1024) verify_combine_exl3(const float* dn, const u8* table, u64 experts, u64 stride, u64 shared0, u32 part, u32 base, const u8* plans,
                                                                       u32 plan_stride, const float* gl, float* y, u32 k, u32 m, u32 hidden, u32 ff) {
    __shared__ float sums[17][128];
    const u32 lane = threadIdx.x & 63, t = threadIdx.x >> 6, ob = blockIdx.x, j = blockIdx.y, li = blockIdx.z;
    const VerifyLayer L = verify_layer(table, li, experts, stride, shared0, part, base);
    const u32 l = L.layer - base, G = m * k, S = G + m, zd = (ff / 128 + 3) / 4;
    const u64 shared = L.shared;
    const u8* pbuf = plans + (u64) l * plan_stride;
    const u32* tidx = (const u32*) pbuf;
    const float* wts = (const float*) (pbuf + G * 4);
    const u32 c = ((const u32*) (pbuf + 2 * G * 4))[j];
    auto finish = [&](bool routed) {
        // everything that does not depend on the expert is requested first, all at once: the partial sums, the weight, the id
        const u32 pair = routed ? j * k + t : G + j;
        float v0 = 0.0f, v1 = 0.0f;
        for (u32 z = 0; z < zd; z++) {
            const float* p = dn + (((u64) li * S + pair) * zd + z) * hidden + ob * 128;
            v0 += p[lane];
            v1 += p[lane + 64];
        }
        const u32 e = routed ? tidx[pair] : 0u;
        const float wt = routed ? wts[pair] : sigmoidf_ref(gl[(u64) l * m + j]);
        if (routed && t >= c) return;
        const u8* down = (const u8*) (routed ? L.experts + e * L.stride : shared) + 2 * (u64) L.part;
        const u16* svh = (const u16*) (down + 2 * (u64) ff) + ob * 128;
        const float s0 = f16_to_f32(svh[lane]), s1 = f16_to_f32(svh[lane + 64]);
        wht128_wave(v0, v1, lane);
        float* o = sums[routed ? t : 16];
        o[lane] = wt * (v0 * s0);
        o[lane + 64] = wt * (v1 * s1);
    };
    if (t < k) finish(true);
    if (shared && t == (k < 16 ? k : 0)) finish(false);
    __syncthreads();
    if (threadIdx.x < 128) {
        float a = 0.0f;
        for (u32 i = 0; i < c; i++) a += sums[i][threadIdx.x];
        if (shared) a += sums[16][threadIdx.x];
        y[((u64) l * m + j) * hidden + ob * 128 + threadIdx.x] = a;
    }
}

// ------------------------------------------------------------------------------------------- one projection for m <= 8 inputs
// y_j = ((x_j * suh) H) W_hat H * svh (matvec_cols_exl3_K, kernels/exl3.cu:260) in two launches: the products of the verify
// layer, 512 inputs and 64 CT columns a workgroup, and the sums' output side.  part: [j][z][out_f].
// grid = (out / (64 CT), ceil(in / 512)), block 256; the inputs are 4 NG at most.
template <int K, bool H, int CT, int NG>
__device__ __forceinline__ void exl3_cols_kernel(const u8* __restrict__ w, const float* __restrict__ x, u32 xs, float* __restrict__ part, u32 in_f, u32 out_f, u32 m) {
    constexpr int NMAX = 4 * NG;
    typedef VerifyRing<K, H, CT> R;
    __shared__ __attribute__((aligned(16))) u32 wb_all[4][R::D * R::UW];
    __shared__ __attribute__((aligned(16))) u16 a_sh[16 * 3 * NMAX * 32];
    __shared__ __attribute__((aligned(16))) float s_mx[4 * NMAX];
    __shared__ float s_iv[NMAX];
    const u32 wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, z = blockIdx.y;
    u64 toks;
    u32 pairs[4];
    verify_shared_item(0, toks, pairs);
    exl3_product<K, H, CT, NG>(w, in_f, out_f, z, [&](u32 r) { return x + (u64) r * xs; }, m, pairs, (u64) gridDim.y * out_f, part + (u64) z * out_f, wave, lane, wb_all[wave], a_sh,
                               s_mx, s_iv);
}

template <int N>
struct ConstInt {
    static constexpr int value = N;
};
// y_j's 128-output block ob: the partial sums added up, the output-side transform, the scales.  A chain of round trips, few waves: of many
// partials sixteen are asked for at once (four at once: a call of 8192 x 16384 at 3 bits for 4 inputs 28.2 us, 26.5, for one 25.9, 23.8; 8192 x
// 2048 at 2 bits 10.4, 9.5; two of 8192 x 32768 at 4 bits 46.6, 45.4).  grid = (out / 128, m), block 64.
extern "C" __global__ void __launch_bounds__(64) exl3_finish_rows(const float* part, const u8* w, float* y, u32 ys, u32 in_f, u32 out_f) {
    const u32 lane = threadIdx.x, ob = blockIdx.x, j = blockIdx.y, zs = (in_f / 128 + 3) / 4;
    const u16* svh = (const u16*) (w + 2 * (u64) in_f) + ob * 128;
    const float s0 = f16_to_f32(svh[lane]), s1 = f16_to_f32(svh[lane + 64]);
    float v0 = 0.0f, v1 = 0.0f;
    // `count` partials' loads in flight together, the last one's again past the end
    auto add = [&](auto count, u32 z0) {
        constexpr int N = decltype(count)::value;
        float a[N][2];
#pragma unroll
        for (int q = 0; q < N; q++) {
            const float* p = part + ((u64) j * zs + min(z0 + q, zs - 1)) * out_f + ob * 128;
            a[q][0] = p[lane];
            a[q][1] = p[lane + 64];
        }
#pragma unroll
        for (int q = 0; q < N; q++)
            if (z0 + q < zs) {
                v0 += a[q][0];
                v1 += a[q][1];
            }
    };
    for (u32 z0 = 0; z0 < zs; z0 += 16) {
        if (zs - z0 > 8) add(ConstInt<16>(), z0);
        else if (zs - z0 > 4) add(ConstInt<8>(), z0);
        else add(ConstInt<4>(), z0);
    }
    wht128_wave(v0, v1, lane);
    float* o = y + (u64) j * ys + ob * 128;
    o[lane] = v0 * s0;
    o[lane + 64] = v1 * s1;
}
#define EXL3_COLS_ENTRIES(K) \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K, 1)) matvec_grouped_exl3_##K(const u8* w, const float* x, u32 xs, float* part, u32 in_f, u32 out_f, u32 m) { \
        exl3_cols_kernel<K, false, 8, 1>(w, x, xs, part, in_f, out_f, m); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K, 1)) matvec_grouped_t4_exl3_##K(const u8* w, const float* x, u32 xs, float* part, u32 in_f, u32 out_f, u32 m) { \
        exl3_cols_kernel<K, false, 4, 1>(w, x, xs, part, in_f, out_f, m); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K, 1)) matvec_grouped_t2_exl3_##K(const u8* w, const float* x, u32 xs, float* part, u32 in_f, u32 out_f, u32 m) { \
        exl3_cols_kernel<K, false, 2, 1>(w, x, xs, part, in_f, out_f, m); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K, 2)) matvec_grouped_w_exl3_##K(const u8* w, const float* x, u32 xs, float* part, u32 in_f, u32 out_f, u32 m) { \
        exl3_cols_kernel<K, false, 8, 2>(w, x, xs, part, in_f, out_f, m); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K, 2)) matvec_grouped_t4w_exl3_##K(const u8* w, const float* x, u32 xs, float* part, u32 in_f, u32 out_f, u32 m) { \
        exl3_cols_kernel<K, false, 4, 2>(w, x, xs, part, in_f, out_f, m); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K, 2)) matvec_grouped_t2w_exl3_##K(const u8* w, const float* x, u32 xs, float* part, u32 in_f, u32 out_f, u32 m) { \
        exl3_cols_kernel<K, false, 2, 2>(w, x, xs, part, in_f, out_f, m); \
    }
#define EXL3_COLS_HALF_ENTRIES(K) \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K + 1, 1)) matvec_grouped_exl3h_##K(const u8* w, const float* x, u32 xs, float* part, u32 in_f, u32 out_f, u32 m) { \
        exl3_cols_kernel<K, true, 8, 1>(w, x, xs, part, in_f, out_f, m); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K + 1, 1)) matvec_grouped_t4_exl3h_##K(const u8* w, const float* x, u32 xs, float* part, u32 in_f, u32 out_f, u32 m) { \
        exl3_cols_kernel<K, true, 4, 1>(w, x, xs, part, in_f, out_f, m); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K + 1, 1)) matvec_grouped_t2_exl3h_##K(const u8* w, const float* x, u32 xs, float* part, u32 in_f, u32 out_f, u32 m) { \
        exl3_cols_kernel<K, true, 2, 1>(w, x, xs, part, in_f, out_f, m); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K + 1, 2)) matvec_grouped_w_exl3h_##K(const u8* w, const float* x, u32 xs, float* part, u32 in_f, u32 out_f, u32 m) { \
        exl3_cols_kernel<K, true, 8, 2>(w, x, xs, part, in_f, out_f, m); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K + 1, 2)) matvec_grouped_t4w_exl3h_##K(const u8* w, const float* x, u32 xs, float* part, u32 in_f, u32 out_f, u32 m) { \
        exl3_cols_kernel<K, true, 4, 2>(w, x, xs, part, in_f, out_f, m); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K + 1, 2)) matvec_grouped_t2w_exl3h_##K(const u8* w, const float* x, u32 xs, float* part, u32 in_f, u32 out_f, u32 m) { \
        exl3_cols_kernel<K, true, 2, 2>(w, x, xs, part, in_f, out_f, m); \
    }
// One column tile a wave, for inputs in 256s (a unit is 16 tile rows).  Above 5 bits a ring holds two units and a weight takes two windows: half the chain
// for a wave of a matrix whose workgroups fill half the chip (a call of 2048 x 4096 at 6 bits for 1, 4 and 8 inputs 8.8, 10.0 and 12.3 us by two tiles, 7.8, 9.1
// and 11.0 by one; at 3 and 4 bits 7.8, 9.0 and 11.3 by either).
#define EXL3_COLS_NARROW_ENTRIES(K) \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K, 1)) matvec_grouped_t1_exl3_##K(const u8* w, const float* x, u32 xs, float* part, u32 in_f, u32 out_f, u32 m) { \
        exl3_cols_kernel<K, false, 1, 1>(w, x, xs, part, in_f, out_f, m); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_VERIFY_OCC(K, 2)) matvec_grouped_t1w_exl3_##K(const u8* w, const float* x, u32 xs, float* part, u32 in_f, u32 out_f, u32 m) { \
        exl3_cols_kernel<K, false, 1, 2>(w, x, xs, part, in_f, out_f, m); \
    }
EXL3_COLS_ENTRIES(1)
EXL3_COLS_ENTRIES(2)
EXL3_COLS_ENTRIES(3)
EXL3_COLS_ENTRIES(4)
EXL3_COLS_ENTRIES(5)
EXL3_COLS_ENTRIES(6)
EXL3_COLS_ENTRIES(7)
EXL3_COLS_ENTRIES(8)
EXL3_COLS_NARROW_ENTRIES(6)
EXL3_COLS_NARROW_ENTRIES(7)
EXL3_COLS_NARROW_ENTRIES(8)
EXL3_COLS_HALF_ENTRIES(1)
EXL3_COLS_HALF_ENTRIES(2)
EXL3_COLS_HALF_ENTRIES(3)

// ------------------------------------------------------------------------------------- the EXL3 head on the matrix cores
// The lm_head of an EXL3 checkpoint (in = hidden, out = vocabulary; kernels/exl3.cu:349-461, 610-625: exl3_rotate_rows_f32 and
// matvec_cols_exl3_pre of the reference) for the m <= 8 rows of a verify batch in one pass over the matrix, with the
// arg-max fused in.  The dot products run on the matrix cores (v_mfma_f32_16x16x16_f16, one a 16 x 16 tile): operand B is
// the tile, a lane supplying 4 CONSECUTIVE weights of the bit stream, which are input rows 2 a, 2 a + 1, 2 a + 8, 2 a + 9
// (a = lane / 16) of output column lane % 16 (exl3.rs:106); their four 16-bit windows lie in the 16 + 3 K stream bits
// that end at bit (t0 + 4) K, t0 = 32 (n % 8) + 8 a + 4 (n / 8): one funnel shift of two ring words (a per-lane constant
// choice) brings them into a register and the windows are then at fixed shifts (two shifts for K > 5).  Operand A is the
// input: row 2 j holds the f16 high part and row 2 j + 1 the f16 low part of token j's rotated input, scaled by the
// power of two that takes the token's largest rotated magnitude to [2^14, 2^15), in the same k order: every product with
// an f16 weight is exact, the matrix core adds in f32, and 8 tokens cost what one costs.
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));

// Launch 1 of the head: token j = blockIdx.x.  Wave w rotates the 128-blocks w, w + waves, .. of x_j (x * suh, the
// transform), the largest magnitude over the row gives the token's scale, and the scaled values go out as f16 high and
// low parts, as the lanes take them: xa[((kb * 4 + t8 / 2) * 64 + 16 (slot / 4) + 2 j + part) * 8 + 4 (t8 % 2) + slot % 4] for tile row t8 of block
// kb; inv[j] undoes the scale.
// grid = m, block = 64 * min(16, in / 128).
#define EXL3_HEAD_NB 4   /* 128-blocks a wave rotates at most: in <= 8192 */
extern "C" __global__ void __launch_bounds__(1024) exl3_head_rotate(const u8* blob, const float* x, u32 xs, u16* xa, float* inv, u32 in_f) {
    __shared__ float s_mx[16];
    const u32 wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, nw = blockDim.x >> 6, j = blockIdx.x;
    const u32 kbs = in_f / 128;
    const u16* suh = (const u16*) blob;
    float rot[EXL3_HEAD_NB][2];
    float mx = 0.0f;
#pragma unroll
    for (int q = 0; q < EXL3_HEAD_NB; q++) {
        const u32 kb = wave + nw * q;
        rot[q][0] = rot[q][1] = 0.0f;
        if (kb < kbs) {
            const float* xj = x + (u64) j * xs + kb * 128;
            float a0 = xj[lane] * f16_to_f32(suh[kb * 128 + lane]), a1 = xj[lane + 64] * f16_to_f32(suh[kb * 128 + 64 + lane]);
            wht128_wave(a0, a1, lane);
            rot[q][0] = a0;
            rot[q][1] = a1;
            mx = fmaxf(mx, fmaxf(__builtin_fabsf(a0), __builtin_fabsf(a1)));
        }
    }
    mx = wave_max_f32(mx);
    if (lane == 0) s_mx[wave] = mx;
    __syncthreads();
    float all = 0.0f;
    for (u32 w = 0; w < nw; w++) all = fmaxf(all, s_mx[w]);
    float scale, iv;
    pow2_scale_of(f32_bits(all), scale, iv);
    if (threadIdx.x == 0) inv[j] = iv;
#pragma unroll
    for (int q = 0; q < EXL3_HEAD_NB; q++) {
        const u32 kb = wave + nw * q;
        if (kb < kbs) {
            u16* blk = xa + (u64) kb * 2048 + 2 * j * 8;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const u32 i = lane + 64 * h;
                const float v = rot[q][h] * scale;
                const _Float16 hi = (_Float16) v;
                const _Float16 lo = (_Float16) (v - (float) hi);
                const u32 t8 = i >> 4, slot = exl3_aslot(i & 15), at = ((t8 >> 1) * 64 + 16 * (slot >> 2)) * 8 + 4 * (t8 & 1) + (slot & 3);
                blk[at] = __builtin_bit_cast(u16, hi);
                blk[at + 8] = __builtin_bit_cast(u16, lo);
            }
        }
    }
}

// Launch 2 of the head: output block ob = blockIdx.x (128 columns of the vocabulary).  Wave w of 4 takes the 128-blocks w, w + 4, .. of the
// input, in units of two tile rows: the trellis and the A rows of a unit come through a ring of two slots.  The four waves' sums
// are added in wave order, scaled back, taken through the output-side transform and scales, optionally stored as logits[j * ls +
// column], and the block's best column of every row goes to part[(ob * 8 + j) * 2] = {value bits, column} (a NaN counts as -inf, ties
// to the lower column).
// With a block list (sel[0] = n, sel[1 ..] = blocks; matvec_cols_exl3_pre_sparse of the reference, exl3.cu tail) workgroup
// i < n takes block sel[1 + i] and its logits and best go to place i instead of ob: logits[j * ls + 128 i + column in block];
// the arithmetic of a block does not depend on which workgroup runs it, so these are the bits the full pass gives.
// Bound by the decode (60 vector cycles for four weights a lane: 41 us of 151936 x 2048 at 4 bits).  Five workgroups a compute unit
// (24 KiB of LDS and 102 registers each), so that the 1187 blocks of that size are one round: 51 us; with all of a wave's A rows in
// LDS three fitted, 1.55 rounds that took two: 57.8 (8 rows of 4096 inputs: the hand-off of the 64 best 199 -> 132 us).  Tried: a
// workgroup of 16 waves a compute unit with its A rows in registers, block after block: 57.8 too, the ends of a block are nobody
// else's time there.
// ONCE: the trellis past the caches, for a head that the last level cannot hold (head_exl3_blocks has the line).  A kernel of its own: the choice
// at every unit cost 1 to 2 %.
// grid = out / 128 (or the list's bound), block 256.
#define EXL3_HEAD_OCC(K) ((K) <= 5 ? 5 : 3)
template <int K, bool ONCE>
__device__ __forceinline__ void exl3_head_kernel(const u8* __restrict__ blob, const u16* __restrict__ xa, const float* __restrict__ inv,
                                                 float* __restrict__ logits, u32 ls, u32* __restrict__ part, u32 in_f, u32 out_f, u32 m,
                                                 const u32* __restrict__ sel) {
    typedef VerifyRing<K, false, 8, 2> R;
    typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
    constexpr int D = R::D, SLOT = R::UW + 256;                             // words of a slot: the unit's tiles, its A rows
    constexpr bool one_shift = 16 + 3 * K <= 32;
    __shared__ __attribute__((aligned(16))) u32 lds[4 * D * SLOT > 4096 ? 4 * D * SLOT : 4096];   // the rings; afterwards the waves' sums [wave][row][128]
    const u32 wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, at = blockIdx.x;
    if (sel && at >= sel[0]) return;                                       // a list shorter than the grid
    const u32 ob = sel ? sel[1 + at] : at;
    const u32 kbs = in_f / 128, total = wave < kbs ? (kbs - wave + 3) / 4 * 4 : 0u;   // this wave's units: four of each of the 128-blocks wave, wave + 4, ..
    const u32 row = lane & 15, a = lane >> 4;
    u32* wb = lds + wave * (D * SLOT);
    const u32 wb_lds = __builtin_amdgcn_readfirstlane(lds_offset(wb));
    const u32 pitch = out_f / 16 * (4 * R::TW);
    const u64 base = uniform_u64((u64) (blob + 2 * (u64) in_f + 2 * (u64) out_f + 4) + (u64) ob * (8 * 4 * R::TW));
    R ring;
    ring.init((const u8*) base, pitch, total, wb_lds, lane);
    auto request = [&](u32 unit, u32 slot) {
        const u32 pair = (wave + (unit & ~3u)) * 4 + (unit & 3);           // of tile rows: 4 (wave + 4 (unit / 4)) + unit % 4
        const u64 from = base + (u64) (2 * pair) * pitch;
#pragma unroll
        for (int i = 0; i < R::NI; i++)
            if (64 * (i + 1) <= 16 * R::CH || 64 * i + lane < 16 * R::CH) lds_load_at<ONCE>(from, ring.off[i], wb_lds + (slot * SLOT + i * 256) * 4);
        lds_load<16>((const u8*) xa + (u64) pair * 1024 + lane * 16, wb_lds + (slot * SLOT + R::UW) * 4);
    };
#pragma unroll
    for (int d = 0; d < D; d++)
        if ((u32) d < total) request(d, d);                                // four units at least, if any
    const u32 t0 = 32 * (row & 7) + 8 * a + 4 * (row >> 3);
    // the 32 stream bits that end at bit e (exclusive) of the tile's ring: word op holds the last of them, word om the rest
    auto window = [&](u32 e, u32& om, u32& op, u32& sh) {
        op = (e - 1) >> 5;
        om = op == 0 ? R::TW - 1 : op - 1;
        sh = 31 - ((e - 1) & 31);
    };
    u32 om1, op1, sh1, om0 = 0, op0 = 0, sh0 = 0;
    window((t0 + 4) * K, om1, op1, sh1);
    if constexpr (!one_shift) window((t0 + 2) * K, om0, op0, sh0);
    f32x4 acc[8];
#pragma unroll
    for (int c = 0; c < 8; c++) acc[c] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    const bool fed = row < 2 * m;                                          // this lane supplies A row `row`
#pragma unroll 1
    for (u32 unit = 0; unit < total; unit++) {
        if (unit + 1 < total) wait_vm<R::NI + 1>();
        else wait_vm<0>();
        const u32* words = wb + (unit & 1) * SLOT;
        u32 w1[16][2], w0[one_shift ? 1 : 16][2];
#pragma unroll
        for (int i = 0; i < 16; i++) {
            w1[i][0] = words[i * R::TW + om1];
            w1[i][1] = words[i * R::TW + op1];
            if constexpr (!one_shift) {
                w0[i][0] = words[i * R::TW + om0];
                w0[i][1] = words[i * R::TW + op0];
            }
        }
        u32x4 av = *(const u32x4*) (words + R::UW + lane * 4);
        if (!fed) av = u32x4{0u, 0u, 0u, 0u};
        if (unit + D < total) {
            __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0): the unit's words are in registers, its slot can take the unit D further on
            request(unit + D, unit & 1);
        }
#pragma unroll
        for (int c = 0; c < 8; c++) {
            u32 b[2][2];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int i = 8 * h + c;
                const u32 top = __builtin_amdgcn_alignbit(w1[i][0], w1[i][1], sh1);
                u32 s0, s1;
                if constexpr (one_shift) {
                    s0 = __builtin_amdgcn_ubfe(top, 3 * K, 16);
                    s1 = __builtin_amdgcn_ubfe(top, 2 * K, 16);
                } else {
                    const u32 low = __builtin_amdgcn_alignbit(w0[i][0], w0[i][1], sh0);
                    s0 = __builtin_amdgcn_ubfe(low, K, 16);
                    s1 = low & 0xffffu;
                }
                const u32 s2 = __builtin_amdgcn_ubfe(top, K, 16), s3 = top & 0xffffu;
                b[h][0] = __builtin_bit_cast(u32, exl3_cb2_pair(s0, s1));
                b[h][1] = __builtin_bit_cast(u32, exl3_cb2_pair(s2, s3));
            }
            const f16x8 bv = __builtin_bit_cast(f16x8, u32x4{b[0][0], b[0][1], b[1][0], b[1][1]});
            acc[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, av), bv, acc[c], 0, 0, 0);
        }
    }
    __syncthreads();                                       // every wave is done with its ring: the space takes the sums
    // D rows 4 a + i: lane group a holds tokens 2 a and 2 a + 1 (high part + low part each)
    float* red = (float*) lds;
    {
        float* o = red + (u64) wave * m * 128;
#pragma unroll
        for (int c = 0; c < 8; c++) {
            if (2 * a < m) o[(2 * a) * 128 + 16 * c + row] = acc[c][0] + acc[c][1];
            if (2 * a + 1 < m) o[(2 * a + 1) * 128 + 16 * c + row] = acc[c][2] + acc[c][3];
        }
    }
    __syncthreads();
    for (u32 j = wave; j < m; j += 4) {
        const u16* svh = (const u16*) (blob + 2 * (u64) in_f) + ob * 128;
        const float sv0 = f16_to_f32(svh[lane]), sv1 = f16_to_f32(svh[lane + 64]);
        float v0 = 0.0f, v1 = 0.0f;
        for (u32 w = 0; w < 4; w++) {
            v0 += red[((u64) w * m + j) * 128 + lane];
            v1 += red[((u64) w * m + j) * 128 + lane + 64];
        }
        const float f = inv[j];
        v0 *= f;
        v1 *= f;
        wht128_wave(v0, v1, lane);
        v0 *= sv0;
        v1 *= sv1;
        const u32 c0 = ob * 128 + lane, c1 = c0 + 64;
        if (logits) {
            logits[(u64) j * ls + at * 128 + lane] = v0;
            logits[(u64) j * ls + at * 128 + lane + 64] = v1;
        }
        float bv = v0 != v0 ? -__builtin_inff() : v0;
        u32 bi = c0;
        argmax_merge(bv, bi, v1 != v1 ? -__builtin_inff() : v1, c1);
#pragma unroll
        for (int h = 1; h < 64; h <<= 1) {
            float ov;
            u32 oi;
            if (h == 1) { ov = lane_xor<1>(bv, lane); oi = f32_bits(lane_xor<1>(bits_f32(bi), lane)); }
            else if (h == 2) { ov = lane_xor<2>(bv, lane); oi = f32_bits(lane_xor<2>(bits_f32(bi), lane)); }
            else if (h == 4) { ov = lane_xor<4>(bv, lane); oi = f32_bits(lane_xor<4>(bits_f32(bi), lane)); }
            else if (h == 8) { ov = lane_xor<8>(bv, lane); oi = f32_bits(lane_xor<8>(bits_f32(bi), lane)); }
            else if (h == 16) { ov = lane_xor<16>(bv, lane); oi = f32_bits(lane_xor<16>(bits_f32(bi), lane)); }
            else { ov = lane_xor<32>(bv, lane); oi = f32_bits(lane_xor<32>(bits_f32(bi), lane)); }
            argmax_merge(bv, bi, ov, oi);
        }
        if (lane == 0) {
            part[((u64) at * 8 + j) * 2] = f32_bits(bv);
            part[((u64) at * 8 + j) * 2 + 1] = bi;
        }
    }
}

// ------------------------------------------------------------------------------------------ the 2-bit screen of the head
// An inexact, optional shortcut of the reference for the top-64 hand-off (exl3.cu:916-987, forward.cu:4371-4497,
// session.rs:5952-5995): a 2-bit copy of the head in the rotated basis scores every output cheaply, only the best 128-output
// blocks are then computed exactly.  Built once a head.  Block (ob, b) = outputs ob * 128 .., inputs b * 128 ..: the decoded
// weights of an input row are transformed over the block's 128 outputs (no 1/sqrt(128) here nor on the inputs: 1/128 once),
// times svh, rounded to f16; an output's 128 values of the block are then cut to the levels {-3, -1, 1, 3} * sh, sh = f16(0.5
// * 0.9957 * rms) (the optimal uniform four-level step of a Gaussian), the level u = 0..3 stored in two bits: the 16-byte
// group [(ob * 2 n_b + 2 b + hb) * 128 + r] holds inputs hb * 64 .. + 63 of output r, word wi bit 8 bi + 2 sl = input
// hb * 64 + 16 wi + 4 sl + bi (a byte lane a dot-product-of-four operand after a shift and a mask).  w_sc[(ob * n_b + b) * 128 + r] = sh.
// grid = (out / 128, in / 128), block 256.
template <int K>
__device__ __forceinline__ void exl3_q2_proxy_build(const u8* __restrict__ blob, u32* __restrict__ w_q2, u16* __restrict__ w_sc, u32 in_f, u32 out_f) {
    __shared__ _Float16 ws[4][16][130];       // a wave's tile row as decoded (f16 values): [input row][output]
    __shared__ u16 wh[128][130];              // the block in the rotated basis as f16: [output][input]
    const u32 wave = threadIdx.x >> 6, lane = threadIdx.x & 63, ob = blockIdx.x, b = blockIdx.y;
    const u32 n_b = in_f / 128, nt = out_f / 16;
    const u32* tr = (const u32*) (blob + 2 * (u64) in_f + 2 * (u64) out_f + 4);
    const u16* svh = (const u16*) (blob + 2 * (u64) in_f) + ob * 128;
    const float sv0 = f16_to_f32(svh[lane]), sv1 = f16_to_f32(svh[lane + 64]);
    const u32 col = (lane >> 3) * 16 + (lane & 7);
    for (u32 kk = wave; kk < 8; kk += 4) {
        u32 S[EXL3_NW(K, false)];
        exl3_load_words<K>(tr, nt, b * 8 + kk, ob, lane, S);
        f16x2 w[16];
        exl3_decode32<K>(S, w);
#pragma unroll
        for (int i = 0; i < 32; i++) ws[wave][EXL3_ROW(i)][col + 8 * EXL3_HALF(i)] = w[i / 2][i % 2];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        for (u32 r = 0; r < 16; r++) {
            float v0 = (float) ws[wave][r][lane], v1 = (float) ws[wave][r][lane + 64];
            wht128_wave_raw(v0, v1, lane);
            // the product rounded to f32 first, then to f16, as the reference's two operations do: left to itself the compiler
            // makes one multiply-and-convert instruction of them, which rounds once and differs where the f32 product is an
            // f16 tie
            float p0 = v0 * 0.0078125f * sv0, p1 = v1 * 0.0078125f * sv1;
            asm volatile("" : "+v"(p0), "+v"(p1));
            wh[lane][kk * 16 + r] = __builtin_bit_cast(u16, (_Float16) p0);
            wh[lane + 64][kk * 16 + r] = __builtin_bit_cast(u16, (_Float16) p1);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    __syncthreads();
    if (threadIdx.x < 128) {
        const u32 r = threadIdx.x;
        float sq = 0.0f;
        for (u32 c = 0; c < 128; c++) {
            const float fv = f16_to_f32(wh[r][c]);
            sq = __builtin_fmaf(fv, fv, sq);
        }
        // the f32 square root correctly rounded, as the reference's sqrtf is: the f64 root of an f32 rounds to it (53 >= 2 * 24 + 2
        // bits); the single-precision instruction is an ulp off now and then
        const float delta = 0.9957f * (float) __builtin_sqrt((double) (sq * 0.0078125f));
        const u16 sh = __builtin_bit_cast(u16, (_Float16) (0.5f * delta));
        const float thr = 2.0f * f16_to_f32(sh);
        w_sc[((u64) ob * n_b + b) * 128 + r] = sh;
        for (u32 hb = 0; hb < 2; hb++) {
            u32x4 words;
#pragma unroll
            for (u32 wi = 0; wi < 4; wi++) {
                u32 pw = 0;
#pragma unroll
                for (u32 sl = 0; sl < 4; sl++)
#pragma unroll
                    for (u32 bi = 0; bi < 4; bi++) {
                        const float fv = f16_to_f32(wh[r][hb * 64 + wi * 16 + sl * 4 + bi]);
                        const u32 q = fv >= 0.0f ? (fv >= thr ? 3u : 2u) : (fv <= -thr ? 0u : 1u);
                        pw |= q << (bi * 8 + sl * 2);
                    }
                words[wi] = pw;
            }
            ((u32x4*) w_q2)[((u64) ob * (n_b * 2) + b * 2 + hb) * 128 + r] = words;
        }
    }
}

// The rows of a batch for the screen (exl3_rotate_rows_f32 + proxy_q2_quant_x of the reference: exl3.cu:610-625,
// forward.cu:4376-4420): block b of row j, (x * suh) transformed without the 1/sqrt(128) factor, as int8 codes with the
// scale amax / 127 (round half to even), four codes a word: xq[(j * n_b + b) * 32 + w] = inputs 4 w .. 4 w + 3 of the block;
// x_sc = the scale, x_corr = -3 * (sum of the codes) * scale (the levels are 2 u - 3 and the screen multiplies by u).
// grid = (in / 128, m), block 64.
extern "C" __global__ void __launch_bounds__(64) proxy_q2_quant_x(const u8* blob, const float* x, u32 xs, u32* xq, float* x_sc, float* x_corr, u32 in_f) {
    const u32 lane = threadIdx.x, b = blockIdx.x, j = blockIdx.y, n_b = in_f / 128;
    const u16* suh = (const u16*) blob + b * 128;
    const float* xj = x + (u64) j * xs + b * 128;
    float v0 = xj[lane] * f16_to_f32(suh[lane]), v1 = xj[lane + 64] * f16_to_f32(suh[lane + 64]);
    wht128_wave_raw(v0, v1, lane);
    const float amax = wave_max_f32(fmaxf(__builtin_fabsf(v0), __builtin_fabsf(v1)));
    const float sc = amax > 0.0f ? amax / 127.0f : 0.0f;
    const float inv = sc > 0.0f ? 1.0f / sc : 0.0f;
    const i32 q0 = (i32) __builtin_rintf(fmaxf(-127.0f, fminf(127.0f, v0 * inv)));
    const i32 q1 = (i32) __builtin_rintf(fmaxf(-127.0f, fminf(127.0f, v1 * inv)));
    u32 p0 = ((u32) q0 & 0xffu) << (8 * (lane & 3)), p1 = ((u32) q1 & 0xffu) << (8 * (lane & 3));
    p0 |= f32_bits(lane_xor<1>(bits_f32(p0), lane));
    p1 |= f32_bits(lane_xor<1>(bits_f32(p1), lane));
    p0 |= f32_bits(lane_xor<2>(bits_f32(p0), lane));
    p1 |= f32_bits(lane_xor<2>(bits_f32(p1), lane));
    u32* o = xq + ((u64) j * n_b + b) * 32;
    if ((lane & 3) == 0) {
        o[lane >> 2] = p0;
        o[16 + (lane >> 2)] = p1;
    }
    i32 tot = q0 + q1;
    tot += (i32) f32_bits(lane_xor<1>(bits_f32((u32) tot), lane));
    tot += (i32) f32_bits(lane_xor<2>(bits_f32((u32) tot), lane));
    tot += (i32) f32_bits(lane_xor<4>(bits_f32((u32) tot), lane));
    tot += (i32) f32_bits(lane_xor<8>(bits_f32((u32) tot), lane));
    tot += (i32) f32_bits(lane_xor<16>(bits_f32((u32) tot), lane));
    tot += (i32) f32_bits(lane_xor<32>(bits_f32((u32) tot), lane));
    if (lane == 0) {
        x_sc[(u64) j * n_b + b] = sc;
        x_corr[(u64) j * n_b + b] = -3.0f * (float) tot * sc;
    }
}

#define EXL3_HEAD_ENTRIES(K) \
    extern "C" __global__ void __launch_bounds__(256, EXL3_HEAD_OCC(K)) head_exl3_##K(const u8* blob, const u16* xa, const float* inv, float* logits, u32 ls, u32* part, u32 in_f, u32 out_f, u32 m, const u32* sel) { \
        exl3_head_kernel<K, false>(blob, xa, inv, logits, ls, part, in_f, out_f, m, sel); \
    } \
    extern "C" __global__ void __launch_bounds__(256, EXL3_HEAD_OCC(K)) head_exl3_past_##K(const u8* blob, const u16* xa, const float* inv, float* logits, u32 ls, u32* part, u32 in_f, u32 out_f, u32 m, const u32* sel) { \
        exl3_head_kernel<K, true>(blob, xa, inv, logits, ls, part, in_f, out_f, m, sel); \
    } \
    extern "C" __global__ void __launch_bounds__(256) exl3_build_q2_proxy_##K(const u8* blob, u32* w_q2, u16* w_sc, u32 in_f, u32 out_f) { \
        exl3_q2_proxy_build<K>(blob, w_q2, w_sc, in_f, out_f); \
    }
EXL3_HEAD_ENTRIES(1)
EXL3_HEAD_ENTRIES(2)
EXL3_HEAD_ENTRIES(3)
EXL3_HEAD_ENTRIES(4)
EXL3_HEAD_ENTRIES(5)
EXL3_HEAD_ENTRIES(6)
EXL3_HEAD_ENTRIES(7)
EXL3_HEAD_ENTRIES(8)

// ------------------------------------------------------------------------ the prefill chunk of an EXL3 layer (matrix cores)
// A chunk's tokens grouped by expert (prefill_group in kernels/prefill.hip: runs of up to 16 XPF_NT (token, rank) pairs of
// one expert are a work item) through gate/up, the activation and down with the item's tokens on the columns of the matrix
// instruction: an expert's weights are decoded once for all tokens of an item (the reference's mma_grouped_exl3_pre_K,
// kernels/exl3.cu:684,704,724, with groups of 64, session.rs:5159-5189).  Every product has the tokens on the columns (operand
// B, lane 16 a + n: token n) and its result on the same lanes as (token n, outputs 4 a .. 4 a + 3).  Inputs ride as single f16
// values after their rotation, scaled by a power of two per token (the reference converts to f16 unscaled); weights are the
// codebook's own f16 values; sums are f32.  Against the exact arithmetic the f16 roundings of the activations cost about 4e-4
// relative L2 of a layer's output (bound of the path: 1e-3).
//
// Three launches a layer.  1 (prefill_rotate_exl3): the inputs of every item through the input sides of its expert's gate and
// up, left as operand rows.  2 (prefill_gate_up_exl3_K): the products over all inputs, both output sides, act = silu(gate) * up and
// its rotation into the down projection's basis, as operand rows again.  3 (prefill_down_exl3_K): the products, the output
// side, the pairs' rows of the layer's result.
// What a token's numbers are does not depend on the item, the workgroup's shape or the other tokens: the sums over the inputs are
// one chain, in the order of the tile rows, and a power of two is a token's (launch 1) or a token's and 128-block's (launch 2).
//
// What bounds it: the decode, 60 vector cycles for four weights a lane, an expert again for every item, and 9 more for each matrix instruction
// (measured: of its 16 cycles a SIMD issues nothing else for 9, whichever wave it comes from), so few, large items; then the ends of a
// workgroup, a third of launch 2's time.  4096 tokens through 512 experts of 2048 x 512 and the shared one at 4 bits, top-10: 130 + 385 +
// 265 us, 568 items and 907 of the down launch, where items of 48 tokens, with every workgroup rotating a quarter of the inputs for itself
// and 738 MB of partial sums in between, took 674 + 213 + 285.  The chunk on inputs that are not in a cache: 1290 -> 914 us.
// Of few items launch 2 is as long as the longest item's chain over all inputs, and the chip is not full: the host takes workgroups of one
// 128-block, two a compute unit, and shorter items, down to one tile, and splits launch 1 and 3 over the 128-blocks (45 tokens at 3 bits 121 -> 100
// us, 512 tokens 273 -> 221, 250 through 32 experts of 3072 x 256, top-3, at 2 bits 104 -> 91 and 159 with items of 128).  Their waves take 32
// columns: with 64 a SIMD had one or two waves, and a wave alone gets a vector instruction in five to eight cycles (16 tokens through 60
// experts of 4096 x 512, top-4, 98 -> 91 us, 64 113 -> 107, 100 through 512 of 2048 x 512, top-10, 122 -> 119; 45 101, 101: 292 such
// workgroups on 256 units, of which some have two and work at the decode's rate).
// Tried: launch 2 by waves of 128 columns for 64 tokens (460 us), its matrix instructions placed among the decode (no change), its two
// waves of a SIMD half a unit apart (2 %), an expert's items on one XCD (less traffic, same time); launch 3 in launch 2's form (272 to 312).

// Most tiles of 16 tokens of a work item: what a wave of 64 columns can keep sums and operands for; in workgroups of one 128-block 4.
#define XPF_NT(K) ((K) <= 5 ? 8 : 6)
#define XPF_NT_N 4
// Units of a wave's ring of trellis rows (64 inputs).  Launch 2, two 128-blocks a workgroup: with six and eight tiles what a compute unit's LDS has
// room for beside three slots of operand rows (XPF_RING); with fewer as many as fit with one slot more, at most 8: an item of one or
// two tiles multiplies little while it waits.  4096 tokens of 512 experts of 2048 x 512, top-10, and the shared one, 4 bits: 916 -> 892
// us (an item of one tile had waited half its time with rings of 3).
// One 128-block: as deep as leaves two workgroups room on a compute unit (rings of 5 units for four tiles and one workgroup a
// unit: 200 tokens of 512 experts of 2048 x 512, top-10, 3 bits 160 us, with rings of 2 and two workgroups 140; with a router without
// preferences 432 and 347).
#define XPF_RING(K) ((K) <= 7 ? 3 : 2)
// (D + 1) 4096 NT + 4096 K D bytes, at most 156 KiB; of one 128-block (D + 1) 4096 NT + 2048 K D, at most 80 KiB
#define XPF_RING_W(K, NT) ((NT) >= 6 ? XPF_RING(K) : (39 - (NT)) / ((NT) + (K)) < 8 ? (39 - (NT)) / ((NT) + (K)) : 8)
#define XPF_RING_N(K, NT) ((40 - 2 * (NT)) / (2 * (NT) + (K)) < 8 ? (40 - 2 * (NT)) / (2 * (NT) + (K)) : 8)
// Launch 3's, of four waves: as deep as leaves two workgroups room with the rows of one tile.
#define XPF_RING_DOWN_N(K) ((K) <= 3 ? 8 : (K) == 4 ? 7 : (K) == 5 ? 5 : (K) <= 7 ? 4 : 3)
// What undoes the 1 / 128 that the stored values carry and applies the transform's 1 / sqrt(128)
#define XPF_UNSCALE 11.3137085f
typedef u16 u16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

// The largest magnitude of the lane's token's 128 values: the lane's 32 of them, then the lanes + 16, + 32, + 48.
__device__ __forceinline__ float xpf_token_max(const f32x4 (&v)[8], u32 lane) {
    float m = 0.0f;
#pragma unroll
    for (int ks = 0; ks < 8; ks++)
#pragma unroll
        for (int q = 0; q < 4; q++) m = fmaxf(m, __builtin_fabsf(v[ks][q]));
    m = fmaxf(m, lane_xor<16>(m, lane));
    return fmaxf(m, lane_xor<32>(m, lane));
}

// The 128-point transform of the lane's token: v[c][q] = value 16 c + 4 a + q (a = lane / 16).  Five of its seven stages are
// between the lane's own registers; the two over the lane number's bits 4 and 5 are swaps of register halves between the lanes
// (one swap serves two registers), after which the lane holds OTHER values of its token: register c, element q is value
// xpf_out_col(c, lane) + q.  Done twice, the values lie as they did at first.
__device__ __forceinline__ u32 xpf_out_col(u32 c, u32 lane) { return 64 * (c >> 2) + 32 * ((lane >> 4) & 1) + 16 * (lane >> 5) + 8 * (c & 1) + 4 * ((c >> 1) & 1); }
__device__ __forceinline__ void xpf_transform(f32x4 (&v)[8]) {
#pragma unroll
    for (int c = 0; c < 8; c++) {
        const float t0 = v[c][0] + v[c][1], t1 = v[c][0] - v[c][1], t2 = v[c][2] + v[c][3], t3 = v[c][2] - v[c][3];
        v[c] = f32x4{t0 + t2, t1 + t3, t0 - t2, t1 - t3};
    }
#pragma unroll
    for (int h = 1; h < 8; h <<= 1)
#pragma unroll
        for (int c = 0; c < 8; c++)
            if (!(c & h)) {
                const f32x4 s = v[c] + v[c + h], d = v[c] - v[c + h];
                v[c] = s;
                v[c + h] = d;
            }
    // lane bit 5 (value bit 3): the upper half of register c and the lower half of register c + 1 change places; then both lanes
    // of a pair hold the two ends of one butterfly.  Register c keeps the sum (bit 3 clear), c + 1 the difference; the lane's
    // bit 5 now says which of the two registers' values (value bit 4) it holds.
#pragma unroll
    for (int c = 0; c < 8; c += 2)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const auto r = __builtin_amdgcn_permlane32_swap(f32_bits(v[c][q]), f32_bits(v[c + 1][q]), false, false);
            v[c][q] = bits_f32(r[0]) + bits_f32(r[1]);
            v[c + 1][q] = bits_f32(r[0]) - bits_f32(r[1]);
        }
    // lane bit 4 (value bit 2) with the registers c and c + 2 (value bit 5) likewise
#pragma unroll
    for (int c = 0; c < 8; c++)
        if (!(c & 2)) {
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const auto r = __builtin_amdgcn_permlane16_swap(f32_bits(v[c][q]), f32_bits(v[c + 2][q]), false, false);
                v[c][q] = bits_f32(r[0]) + bits_f32(r[1]);
                v[c + 2][q] = bits_f32(r[0]) - bits_f32(r[1]);
            }
        }
}

// The operand rows of 16 tokens and one 128-block: a 32-deep matrix instruction takes two tile rows, lane 16 a + n holds of either the
// inputs 2 a, 2 a + 1, 2 a + 8, 2 a + 9 of token n (the order in which the decode yields weights).  [pair of tile rows][lane][8], as the
// lanes read them: 4 KiB, in two halves of 64 inputs half_step u16 apart.
#define XPF_ROWS_U16 2048
#define XPF_HALF_U16 1024     // of the first or the last 64 inputs: how the operand rows are laid out, [64-block][tile]
__device__ __forceinline__ u32 xpf_f16_pair(float a, float b) { return __builtin_bit_cast(u32, f16x2{(_Float16) a, (_Float16) b}); }
// The values after one transform (xpf_out_col): a lane holds whole tile rows; the lanes 32 on hold the other row of each pair.
__device__ __forceinline__ void xpf_put_transformed(u16* rows, u32 half_step, const f32x4 (&v)[8], u32 lane) {
    const u32 n = lane & 15, b4 = (lane >> 4) & 1, b5 = lane >> 5;
#pragma unroll
    for (u32 h = 0; h < 2; h++)
#pragma unroll
        for (u32 a = 0; a < 2; a++) {
            u32 w[2][2];
#pragma unroll
            for (u32 j = 0; j < 2; j++) {
                // words of place a (register 4 h + j, elements 2 a, 2 a + 1) and of place a + 2 (register 4 h + 2 + j)
                const auto r = __builtin_amdgcn_permlane32_swap(xpf_f16_pair(v[4 * h + j][2 * a], v[4 * h + j][2 * a + 1]), xpf_f16_pair(v[4 * h + 2 + j][2 * a], v[4 * h + 2 + j][2 * a + 1]), false, false);
                w[0][j] = r[0];
                w[1][j] = r[1];
            }
            const u32x4 o = {w[0][0], w[0][1], w[1][0], w[1][1]};
            __builtin_nontemporal_store(o, (u32x4*) (rows + h * half_step + ((b4 * 4 + a + 2 * b5) * 16 + n) * 8));
        }
}
// The values as they lie before a transform or after two.
__device__ __forceinline__ void xpf_put_plain(u16* rows, u32 half_step, const f32x4 (&v)[8], u32 lane) {
    const u32 n = lane & 15, b4 = (lane >> 4) & 1, b5 = lane >> 5;
#pragma unroll
    for (u32 p = 0; p < 4; p++) {
        u32 w[2][2];
#pragma unroll
        for (u32 h = 0; h < 2; h++) {
            const auto r = __builtin_amdgcn_permlane32_swap(xpf_f16_pair(v[2 * p + h][0], v[2 * p + h][1]), xpf_f16_pair(v[2 * p + h][2], v[2 * p + h][3]), false, false);
            w[h][0] = r[0];
            w[h][1] = r[1];
        }
        *(u32x4*) (rows + (p >> 1) * half_step + (((p & 1) * 4 + 2 * b4 + b5) * 16 + n) * 8) = u32x4{w[0][0], w[0][1], w[1][0], w[1][1]};
    }
}

// An item: its expert (ne: the shared one), the number n of its pairs (0: there is no such item), its first pair's place in `list`, its
// tiles of 16 tokens and the number of the first of them: the operand rows lie behind each other by tiles, an expert's from a place on
// that its first pair's and its number tell.
struct XpfItem {
    u32 e, n, first, tiles, base;
};
__device__ __forceinline__ XpfItem xpf_item(const u32* __restrict__ offs, const u32* __restrict__ items, u32 item, u32 ne, bool has_shared, u32 tok) {
    XpfItem it{0, 0, 0, 0, 0};
    if (item >= items[0]) return it;
    it.e = items[1 + 2 * item];
    if (it.e == ne && !has_shared) return it;
    it.first = offs[it.e] + items[2 + 2 * item];
    it.n = min(tok, offs[it.e + 1] - it.first);
    it.tiles = (it.n + 15) / 16;
    it.base = offs[it.e] / 16 + it.e + items[2 + 2 * item] / 16;
    return it;
}
// The item of a workgroup of a launch of 8 ceil(bound / 8) parts workgroups, and which of the item's parts it takes.  Workgroup i runs on
// XCD i mod 8: the parts of an item follow each other on one of them, so that its operand rows come from memory once.
__device__ __forceinline__ u32 xpf_place(u32 parts, u32& part) {
    part = blockIdx.x / 8 % parts;
    return blockIdx.x / 8 / parts * 8 + (blockIdx.x & 7);
}
// The products are compiled for 1, 2, 4, 6 and 8 token tiles: an item of 3, 5 or 7 has the next one's do for it, the last tile's
// operand rows being whatever lies there.
template <int MOST, class F>
__device__ __forceinline__ void xpf_tiles(u32 tiles, F&& run) {
    if (tiles == 1) return run(ConstInt<1>());
    if (tiles == 2) return run(ConstInt<2>());
    if constexpr (MOST > 6) {
        if (tiles > 6) return run(ConstInt<8>());
    }
    if constexpr (MOST > 4) {
        if (tiles > 4) return run(ConstInt<6>());
    }
    run(ConstInt<4>());
}

// Launch 1: a tile (16 tokens) of an item and one of `shares` of the inputs' 128-blocks: wave w takes 4 share + w, from there 4 shares on, ..  A token's power of two takes a bound
// of its inputs times the projection's input scales to [2^7, 2^8): no value passes 2^15 in the transform.  Values 2^21 below the bound are
// f16's subnormals, whose last bit is 2^31 below it.  The bound is the largest input (most, from the routing launch) times the largest
// scale where all scales, or those of the four channels about that input, are within 2^10 of the largest, so that the bound is no further than
// that from the largest product; else (a large input of a channel that the expert scales to next to nothing) the largest product, which
// takes another pass over the inputs (such a pass for every token: 52 us of 4096 tokens' 920, 4 of 45 tokens' 121).
// rows: an item's [gate, up][64-block][tile], inv: [gate, up][tile][16].
// Bound by the rows it writes (8 bytes an input and pair), past the caches: the next launch begins with rows that were written long before (kept there:
// 4096 tokens as above 857 us for the chunk, 844, 512 tokens 220, 218.5, 100 tokens 119, 118, 250 through 32 experts 84, 83).
// grid = xpf_place's, of `tiles * shares` parts, block 256.
extern "C" __global__ void __launch_bounds__(256) prefill_rotate_exl3(const u64* eaddr, const u64* sh_addr, const u32* offs, const u32* list, const u32* items, const float* x,
                                                                      const u32* most, u16* rows, float* inv, u32 ne, u32 k, u32 npairs, u32 hidden, u32 tok, u32 tiles, u32 shares) {
    __shared__ u32 s_scale[2][4], s_least[2][4];
    __shared__ float s_most[2][4][16];
    const u32 wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, kbs = hidden / 128;
    u32 part;
    const u32 item = xpf_place(tiles * shares, part), T = part / shares, share = part - T * shares, first = share * 4 + wave;
    const XpfItem it = xpf_item(offs, items, item, ne, sh_addr != nullptr, tok);
    if (T >= it.tiles) return;
    const u32 e = it.e, pair = list[it.first + min(16 * T + (lane & 15), it.n - 1)];   // places past the item's end repeat its last pair: nothing reads them
    const u32 token = pair < npairs ? pair / k : pair - npairs;
    const float am = bits_f32(most[2 * token]);
    const u16* suh[2] = {(const u16*) (e < ne ? eaddr[e] : sh_addr[0]), (const u16*) (e < ne ? eaddr[(u64) ne + e] : sh_addr[1])};
#pragma unroll
    for (int s = 0; s < 2; s++) {
        u32 m = 0, l = 0x7fffu;
        for (u32 i = threadIdx.x; i < hidden / 8; i += 256) {
            const u32x4a v = ((const u32x4a*) suh[s])[i];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                m = max(m, max(v[q] & 0x7fffu, (v[q] >> 16) & 0x7fffu));
                l = min(l, min(v[q] & 0x7fffu, (v[q] >> 16) & 0x7fffu));
            }
        }
        m = wave_max_u32(m);
        l = wave_min_u32(l);
        if (lane == 0) {
            s_scale[s][wave] = m;
            s_least[s][wave] = l;
        }
    }
    const float* xr = x + (u64) token * hidden + 4 * (lane >> 4);
    f32x4 xv[8];
    auto inputs = [&](u32 kb) {
#pragma unroll
        for (int ks = 0; ks < 8; ks++) xv[ks] = *(const f32x4*) (xr + kb * 128 + 16 * ks);
    };
    inputs(min(first, kbs - 1));   // on their way while the scales' maxima are made
    __syncthreads();
    // a block's inputs times their scales
    auto scaled = [&](u32 s, u32 kb, f32x4 (&v)[8]) {
#pragma unroll
        for (int ks = 0; ks < 8; ks++) {
            const u16x4 s4 = *(const u16x4*) (suh[s] + kb * 128 + 16 * ks + 4 * (lane >> 4));
#pragma unroll
            for (int q = 0; q < 4; q++) v[ks][q] = xv[ks][q] * f16_to_f32(s4[q]);
        }
    };
    float bound[2], scale[2], largest[2];
    bool wide = false;   // scales further apart
#pragma unroll
    for (int s = 0; s < 2; s++) {
        largest[s] = f16_to_f32((u16) max(max(s_scale[s][0], s_scale[s][1]), max(s_scale[s][2], s_scale[s][3])));
        wide = wide || f16_to_f32((u16) min(min(s_least[s][0], s_least[s][1]), min(s_least[s][2], s_least[s][3]))) * 0x1p10f < largest[s];
        bound[s] = am * largest[s];
    }
    bool loose[2] = {false, false};
    if (__builtin_amdgcn_ballot_w64(wide)) {
        const u32 at = most[2 * token + 1];
#pragma unroll
        for (int s = 0; s < 2; s++) {
            const u16x4 own = *(const u16x4*) (suh[s] + at) & (u16) 0x7fff;
            loose[s] = f16_to_f32(min(min(own[0], own[1]), min(own[2], own[3]))) * 0x1p10f < largest[s];
        }
    }
    if (__builtin_amdgcn_ballot_w64(loose[0] || loose[1])) {   // the same in all four waves
        float p[2] = {0.0f, 0.0f};
#pragma unroll 1
        for (u32 kb = wave; kb < kbs; kb += 4) {
            f32x4 v[8];
            inputs(kb);
#pragma unroll
            for (int s = 0; s < 2; s++) {
                scaled(s, kb, v);
                p[s] = fmaxf(p[s], xpf_token_max(v, lane));
            }
        }
#pragma unroll
        for (int s = 0; s < 2; s++)
            if (lane < 16) s_most[s][wave][lane] = p[s];
        inputs(min(first, kbs - 1));
        __syncthreads();
#pragma unroll
        for (int s = 0; s < 2; s++) {
            const u32 t = lane & 15;
            if (loose[s]) bound[s] = fmaxf(fmaxf(s_most[s][0][t], s_most[s][1][t]), fmaxf(s_most[s][2][t], s_most[s][3][t]));
        }
    }
#pragma unroll
    for (int s = 0; s < 2; s++) {
        float iv;
        pow2_scale_of(f32_bits(bound[s]), scale[s], iv);
        scale[s] *= 0.0078125f;
        if (first == 0 && lane < 16) inv[(it.base * 2 + s * it.tiles + T) * 16 + lane] = iv * XPF_UNSCALE;
    }
    for (u32 kb = first; kb < kbs; kb += 4 * shares) {
        if (kb != first) inputs(kb);
#pragma unroll
        for (int s = 0; s < 2; s++) {
            f32x4 v[8];
            scaled(s, kb, v);
#pragma unroll
            for (int ks = 0; ks < 8; ks++) v[ks] *= scale[s];
            xpf_transform(v);
            xpf_put_transformed(rows + ((u64) it.base * 2 + s * it.tiles) * kbs * XPF_ROWS_U16 + (2 * kb * it.tiles + T) * XPF_HALF_U16, it.tiles * XPF_HALF_U16, v, lane);
        }
    }
}

// What a wave multiplies at a time: two tile rows of four (CT = 2: two) column tiles (the words of their windows) with the operand rows of NT token
// tiles, `step` u16 from one to the next.  read() and rows() ask LDS for them, products() adds acc[T][c][q] = output 16 c + 4 a + q of token 16 T + n.
template <int K, int CT, int NT>
struct XpfStep {
    static constexpr int TW = EXL3_TILE_WORDS(K, false);
    static constexpr bool one_shift = 16 + 3 * K <= 32;
    static constexpr int W = CT < 4 ? CT : 4;   // column tiles of a step
    u32 w1[2 * W][2], w0[one_shift ? 1 : 2 * W][2];
    static __device__ __forceinline__ void window(u32 e, u32& om, u32& op, u32& sh) {
        op = (e - 1) >> 5;
        om = op == 0 ? TW - 1 : op - 1;
        sh = 31 - ((e - 1) & 31);
    }
    static __device__ __forceinline__ u32 first(u32 lane) { return 32 * (lane & 7) + 8 * (lane >> 4) + 4 * ((lane & 15) >> 3); }   // the lane's first weight
    // step s of the unit at `row`: its tile rows 2 s and 2 s + 1 (CT = 4, 2: the unit has four), or their column tiles 4 s .. 4 s + 3 (CT = 8)
    __device__ __forceinline__ void read(const u32* row, u32 s, u32 lane) {
        u32 om, op, sh;
        row += s * (CT == 8 ? 4 : 2 * CT) * TW;
        window((first(lane) + 4) * K, om, op, sh);
#pragma unroll
        for (int i = 0; i < 2 * W; i++) {
            w1[i][0] = row[(i / W * CT + i % W) * TW + om];
            w1[i][1] = row[(i / W * CT + i % W) * TW + op];
        }
        if constexpr (!one_shift) {
            window((first(lane) + 2) * K, om, op, sh);
#pragma unroll
            for (int i = 0; i < 2 * W; i++) {
                w0[i][0] = row[(i / W * CT + i % W) * TW + om];
                w0[i][1] = row[(i / W * CT + i % W) * TW + op];
            }
        }
    }
    static __device__ __forceinline__ void rows(u32x4 (&xv)[NT], const u16* xa, u32 step) {
#pragma unroll
        for (int T = 0; T < NT; T++) xv[T] = *(const u32x4*) (xa + T * step);
    }
    // adds to acc[T][c0 ..]
    template <int c0>
    __device__ __forceinline__ void products(const u32x4 (&xv)[NT], f32x4 (&acc)[NT][CT], u32 lane) const {
        u32 om, op, sh1, sh0 = 0;
        window((first(lane) + 4) * K, om, op, sh1);
        if constexpr (!one_shift) window((first(lane) + 2) * K, om, op, sh0);
#pragma unroll
        for (int c = 0; c < W; c++) {
            u32 b[2][2];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int i = W * h + c;
                const u32 hi = __builtin_amdgcn_alignbit(w1[i][0], w1[i][1], sh1);
                u32 s0, s1;
                if constexpr (one_shift) {
                    s0 = __builtin_amdgcn_ubfe(hi, 3 * K, 16);
                    s1 = __builtin_amdgcn_ubfe(hi, 2 * K, 16);
                } else {
                    const u32 lo = __builtin_amdgcn_alignbit(w0[i][0], w0[i][1], sh0);
                    s0 = __builtin_amdgcn_ubfe(lo, K, 16);
                    s1 = lo & 0xffffu;
                }
                const u32 s2 = __builtin_amdgcn_ubfe(hi, K, 16), s3 = hi & 0xffffu;
                b[h][0] = __builtin_bit_cast(u32, exl3_cb2_pair(s0, s1));
                b[h][1] = __builtin_bit_cast(u32, exl3_cb2_pair(s2, s3));
            }
            const f16x8 bv = __builtin_bit_cast(f16x8, u32x4{b[0][0], b[0][1], b[1][0], b[1][1]});
#pragma unroll
            for (int T = 0; T < NT; T++) acc[T][c0 + c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bv, __builtin_bit_cast(f16x8, xv[T]), acc[T][c0 + c], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
};

// The products of a wave (64 columns) over the `ring.units` 64-blocks of the inputs.  The operand rows (src: [64-block][tiles], whole
// item) come through a ring of NB slots of NT tiles in LDS (`stage`, slots `slot_u16` apart) that the NW waves of one projection share, of
// which this is number `part`: requested NB - 1 units ahead, each wave its share, a barrier a unit.  The waits count the loads that every wave makes of a
// unit: where its operand rows do not divide evenly (one tile: two loads for four waves) a wave that makes one more waits for as many loads as units are in
// flight sooner than it would have to, and the others with it at the barrier.  A step's words and
// operand rows are read while the one before is multiplied. The whole workgroup calls this with the same number of units.  D + 1 >= NB.
template <int K, int NT, int NB, int NW, class R>
__device__ __forceinline__ void xpf_stream(const R& ring, const u32* wb, const u16* __restrict__ src, u16* stage, u32 slot_u16, u32 tiles, u32 part, u32 lane,
                                           f32x4 (&acc)[NT][4]) {
    constexpr int D = R::D, LEAST = NT <= 2 ? NT : NT - 1, A = 2 * LEAST / NW;   // A: loads of a unit's operand rows that every wave makes at least
    static_assert(D + 1 >= NB && R::UR == 4, "operand rows are requested no earlier than the trellis rows of their unit");
    auto request = [&](u32 unit, u32 slot) {
        const u8* from = (const u8*) (src + (u64) unit * tiles * XPF_HALF_U16) + lane * 16;
        const u32 to = __builtin_amdgcn_readfirstlane(lds_offset(stage + slot * slot_u16));
        for (u32 i = part; i < 2 * tiles; i += NW) lds_load<16>(from + i * 1024, to + i * 1024);
    };
#pragma unroll
    for (int T = 0; T < NT; T++)
#pragma unroll
        for (int c = 0; c < 4; c++) acc[T][c] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int i = -D; i < 0; i++) {
        // a stream may be shorter than its ring (hidden = 256: four units)
        if ((u32) (i + D) < ring.units) ring.issue(i + D, i + D, lane);
        if (i + NB - 1 >= 0 && (u32) (i + NB - 1) < ring.units) request(i + NB - 1, i + NB - 1);
    }
    // this wave's share of a unit's operand rows has landed (behind it: NB - 2 times a unit's trellis rows and operand rows, but for the
    // stream's end); every wave's, and the slot of the unit before has been read
    auto ready = [&](u32 unit) {
        if (unit + D <= ring.units) wait_vm<(NB - 2) * (R::NI + A)>();
        else wait_vm<0>();
        lds_barrier();
    };
    typedef XpfStep<K, 4, NT> Step;
    Step s0, s1;
    u32x4 x0[NT], x1[NT];
    ready(0);
    s0.read(wb, 0, lane);
    Step::rows(x0, stage + lane * 8, XPF_HALF_U16);
    u32 slot = 0, at = 0;
#pragma unroll 1
    for (u32 unit = 0; unit < ring.units; unit++) {
        s1.read(wb + slot * R::UW, 1, lane);
        Step::rows(x1, stage + at * slot_u16 + 512 + lane * 8, XPF_HALF_U16);
        __builtin_amdgcn_sched_barrier(0);
        s0.template products<0>(x0, acc, lane);
        __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0): the unit's words are in registers, its slot can take the unit D further on
        if (unit + D < ring.units) ring.issue(unit + D, slot, lane);
        if (unit + NB - 1 < ring.units) request(unit + NB - 1, at == 0 ? NB - 1 : at - 1);
        slot = slot + 1 == (u32) D ? 0u : slot + 1;
        at = at + 1 == (u32) NB ? 0u : at + 1;
        if (unit + 1 < ring.units) {
            ready(unit + 1);
            s0.read(wb + slot * R::UW, 0, lane);
            Step::rows(x0, stage + at * slot_u16 + lane * 8, XPF_HALF_U16);
            __builtin_amdgcn_sched_barrier(0);
        }
        s1.template products<0>(x1, acc, lane);
    }
}

// The same for waves of 32 columns, four to a projection: a unit has half the tiles and the waves of a compute unit are twice as many.  For short
// chunks, whose items leave a SIMD one or two waves of 64 columns: such a wave spends half of its time on what comes between the decodes.
template <int K, int NT, int NB, class R>
__device__ __forceinline__ void xpf_stream_n(const R& ring, const u32* wb, const u16* __restrict__ src, u16* stage, u32 slot_u16, u32 tiles, u32 part, u32 lane, f32x4 (&acc)[NT][2]) {
    constexpr int D = R::D, LEAST = NT <= 2 ? NT : NT - 1, A = 2 * LEAST / 4;   // A: loads of a unit's operand rows that every wave makes at least
    static_assert(D + 1 >= NB && R::UR == 4, "operand rows are requested no earlier than the trellis rows of their unit");
    auto request = [&](u32 unit, u32 slot) {
        const u8* from = (const u8*) (src + (u64) unit * tiles * XPF_HALF_U16) + lane * 16;
        const u32 to = __builtin_amdgcn_readfirstlane(lds_offset(stage + slot * slot_u16));
        for (u32 i = part; i < 2 * tiles; i += 4) lds_load<16>(from + i * 1024, to + i * 1024);
    };
#pragma unroll
    for (int T = 0; T < NT; T++) acc[T][0] = acc[T][1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int i = -D; i < 0; i++) {
        if ((u32) (i + D) < ring.units) ring.issue(i + D, i + D, lane);
        if (i + NB - 1 >= 0 && (u32) (i + NB - 1) < ring.units) request(i + NB - 1, i + NB - 1);
    }
    auto ready = [&](u32 unit) {
        if (unit + D <= ring.units) wait_vm<(NB - 2) * (R::NI + A)>();
        else wait_vm<0>();
        lds_barrier();
    };
    typedef XpfStep<K, 2, NT> Step;
    Step s0, s1;
    u32x4 x0[NT], x1[NT];
    ready(0);
    s0.read(wb, 0, lane);
    Step::rows(x0, stage + lane * 8, XPF_HALF_U16);
    u32 slot = 0, at = 0;
#pragma unroll 1
    for (u32 unit = 0; unit < ring.units; unit++) {
        s1.read(wb + slot * R::UW, 1, lane);
        Step::rows(x1, stage + at * slot_u16 + 512 + lane * 8, XPF_HALF_U16);
        __builtin_amdgcn_sched_barrier(0);
        s0.template products<0>(x0, acc, lane);
        __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0): the unit's words are in registers, its slot can take the unit D further on
        if (unit + D < ring.units) ring.issue(unit + D, slot, lane);
        if (unit + NB - 1 < ring.units) request(unit + NB - 1, at == 0 ? NB - 1 : at - 1);
        slot = slot + 1 == (u32) D ? 0u : slot + 1;
        at = at + 1 == (u32) NB ? 0u : at + 1;
        if (unit + 1 < ring.units) {
            ready(unit + 1);
            s0.read(wb + slot * R::UW, 0, lane);
            Step::rows(x0, stage + at * slot_u16 + lane * 8, XPF_HALF_U16);
            __builtin_amdgcn_sched_barrier(0);
        }
        s1.template products<0>(x1, acc, lane);
    }
}

// What launch 2 makes of a token tile's sums over the inputs (g, u: gate and up of a 128-block, in true units but for the output side):
// output sides, act = silu(gate) * up times the down projection's input scales, its rotation, as operand rows.  The token's power of
// two for this block is a multiple of 8 in the exponent, so that blocks mostly share one; inv undoes it.
__device__ __forceinline__ void xpf_activate(f32x4 (&g)[8], f32x4 (&u)[8], const u16* svg, const u16* svu, const u16* suh, u16* rows, u32 half_step, float* inv, u32 lane) {
    xpf_transform(g);
    xpf_transform(u);
#pragma unroll
    for (int c = 0; c < 8; c++) {
        const u32 at = xpf_out_col(c, lane);
        const u16x4 a4 = *(const u16x4*) (svg + at), b4 = *(const u16x4*) (svu + at), c4 = *(const u16x4*) (suh + at);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const float gate = g[c][q] * (f16_to_f32(a4[q]) * 0.08838835f), up = u[c][q] * (f16_to_f32(b4[q]) * 0.08838835f);
            g[c][q] = (siluf_ref(gate) * up) * f16_to_f32(c4[q]);
        }
    }
    float scale, all;
    pow2_scale_of(f32_bits(xpf_token_max(g, lane)), scale, all);
    const u32 sb = max((f32_bits(scale) >> 23) & ~7u, 8u);
    scale = bits_f32(sb << 23) * 0.0078125f;
    if (lane < 16) inv[lane] = bits_f32((254u - sb) << 23) * XPF_UNSCALE;
#pragma unroll
    for (int c = 0; c < 8; c++) g[c] *= scale;
    xpf_transform(g);
    xpf_put_plain(rows, half_step, g, lane);
}

// A token's factors (what undoes its blocks' powers of two, `f[16 b]`) as launch 3 may take its sums from one block's power of two to the
// next one's.  The sums of a block are below 2^25 in its own units (128 inputs of at most 2^15 times weights below 4), whatever follows
// multiplies them by f[b - 1] / f[b], and what counts is the product of these steps from the largest factor before a block to its own: at
// most 2^88 keeps four blocks' sums below 2^116.  A block beyond that is nothing beside the sums (its values are below 2^-80 of the
// largest ones): drop(b) makes it zeros, and it takes the factor of the one before.
template <class Drop>
__device__ __forceinline__ void xpf_chain(float* f, u32 fbs, Drop drop) {
    float most = f[0], last = most;
    for (u32 b = 1; b < fbs; b++) {
        const float here = f[16 * b];
        if (most > here * 0x1p88f) {
            f[16 * b] = last;
            drop(b);
        } else {
            last = here;
            most = fmaxf(most, here);
        }
    }
}

// A workgroup's sums came through LDS (x: [block of 128 columns][of R tiles][register][lane]), so that a wave has all 128 columns of a
// token tile.
__device__ __forceinline__ void xpf_take(const f32x4* x, u32 place, f32x4 (&v)[8], u32 lane) {
#pragma unroll
    for (u32 c = 0; c < 8; c++) v[c] = x[(place * 8 + c) * 64 + lane];
}

// Launch 2: an item (of up to tok pairs) and NCB 128-column blocks of ff: two, with two waves a projection and block (NCB = 2), or one, with four.  rows2:
// [tile][128-block of ff], inv2: [tile][128-block][16].  grid = xpf_place's, of ff / 128 / NCB parts, block 512; dynamic LDS: NB
// slots of two projections' NT tiles and the waves' rings (for the NT of 1, 2, 4, 6, 8 that takes most), or the exchange of the sums, 64
// KiB NCB for four tiles.
template <int K, int NCB>
__device__ __forceinline__ void prefill_gate_up_exl3_kernel(const u64* __restrict__ eaddr, const u64* __restrict__ sh_addr, const u32* __restrict__ offs, const u32* __restrict__ items,
                                                            const u16* __restrict__ rows, const float* __restrict__ inv, u16* __restrict__ rows2, float* __restrict__ inv2, u32 ne, u32 hidden,
                                                            u32 ff, u32 tok) {
    extern __shared__ __attribute__((aligned(16))) u32 dyn[];
    constexpr int CT = NCB == 2 ? 4 : 2;   // column tiles a wave
    const u32 wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const u32 sel = wave / 4, part = wave % 4, b = NCB == 2 ? part / 2 : 0, at = NCB == 2 ? part & 1 : part;   // at: which of the block's waves
    const u32 kbs = hidden / 128, fbs = ff / 128;
    u32 group;
    const u32 item = xpf_place(fbs / NCB, group), cb = group * NCB + b;
    const XpfItem it = xpf_item(offs, items, item, ne, sh_addr != nullptr, tok);
    if (it.n == 0) return;
    const u32 e = it.e;
    const u8* bg = (const u8*) (e < ne ? eaddr[e] : sh_addr[0]);
    const u8* bu = (const u8*) (e < ne ? eaddr[(u64) ne + e] : sh_addr[1]);
    const u8* bd = (const u8*) (e < ne ? eaddr[2ull * ne + e] : sh_addr[2]);
    xpf_tiles<NCB == 2 ? XPF_NT(K) : XPF_NT_N>(it.tiles, [&](auto n) {
        constexpr int NT = decltype(n)::value, G = NT < 4 ? NT : 4;
        typedef VerifyRing<K, false, CT, NCB == 2 ? XPF_RING_W(K, NT) : XPF_RING_N(K, NT), 4 * CT, false> R;
        constexpr int NB = NCB == 2 && NT >= 6 ? 3 : R::D + 1;
        u32* wb = dyn + NB * 2 * NT * (XPF_HALF_U16 / 2) + wave * (R::D * R::UW);
        R ring;
        ring.init((sel ? bu : bg) + 2 * (u64) hidden + 2 * (u64) ff + 4 + (u64) (cb * 8 + at * CT) * (4 * R::TW), (ff / 16) * (4 * R::TW), 2 * kbs,
                  __builtin_amdgcn_readfirstlane(lds_offset(wb)), lane);
        f32x4 acc[NT][CT];
        const u16* src = rows + ((u64) it.base * 2 + sel * it.tiles) * kbs * XPF_ROWS_U16;
        u16* stage = (u16*) dyn + sel * NT * XPF_HALF_U16;
        if constexpr (NCB == 2) xpf_stream<K, NT, NB, 4>(ring, wb, src, stage, 2 * NT * XPF_HALF_U16, it.tiles, part, lane, acc);
        else xpf_stream_n<K, NT, NB>(ring, wb, src, stage, 2 * NT * XPF_HALF_U16, it.tiles, part, lane, acc);
        const float* iv = inv + (it.base * 2 + sel * it.tiles) * 16 + (lane & 15);
        f32x4* x = (f32x4*) dyn;
#pragma unroll
        for (int T0 = 0; T0 < NT; T0 += G) {
            lds_barrier();
#pragma unroll
            for (int i = 0; i < G && T0 + i < NT; i++) {
                const float f = iv[16 * min((u32) (T0 + i), it.tiles - 1)];
#pragma unroll
                for (int c = 0; c < CT; c++) {
                    acc[T0 + i][c] *= f;
                    x[(((b * 2 + sel) * G + i) * 8 + at * CT + c) * 64 + lane] = acc[T0 + i][c];
                }
            }
            lds_barrier();
            // a wave a tile and block
            const u32 i = NCB == 2 ? part - 2 * b + 2 * sel : wave, T = T0 + i;
            if (i < (u32) G && T < it.tiles) {
                f32x4 g[8], u[8];
                xpf_take(x, (b * 2) * G + i, g, lane);
                xpf_take(x, (b * 2 + 1) * G + i, u, lane);
                xpf_activate(g, u, (const u16*) (bg + 2 * (u64) hidden) + cb * 128, (const u16*) (bu + 2 * (u64) hidden) + cb * 128, (const u16*) bd + cb * 128,
                             rows2 + ((u64) (it.base + T) * fbs + cb) * XPF_ROWS_U16, XPF_HALF_U16, inv2 + ((it.base + T) * fbs + cb) * 16, lane);
            }
        }
    });
}

// Launch 3: an item of up to ntl (at most XPF_DOWN_NT) tiles and one of `parts` shares of the 128-column blocks of hidden, a wave a block at a time: the
// products of the item's operand rows over ff and the output side: eo[pair][hidden].  The rows, their factors and the output scales are copied
// to LDS once; from then on every wave goes its own way, its ring of trellis rows filled from one block to the next.
// grid = xpf_place's, block 64 W; dynamic LDS in words: ntl tiles' rows (fbs * 1024 each), factors (fbs * 16 each), 64
// XPF_DOWN_BLOCKS a wave for the output scales, the waves' rings.
#define XPF_DOWN_NT 4
#define XPF_DOWN_BLOCKS 4   /* most column blocks of a wave: parts * W * 4 >= hidden / 128 */
template <int K, int DEPTH>
__device__ __forceinline__ void prefill_down_exl3_kernel(const u64* __restrict__ eaddr, const u64* __restrict__ sh_addr, const u32* __restrict__ offs, const u32* __restrict__ list,
                                                         const u32* __restrict__ items, const u16* __restrict__ rows, const float* __restrict__ inv, float* __restrict__ eo, u32 ne, u32 hidden,
                                                         u32 ff, u32 ntl, u32 parts) {
    typedef VerifyRing<K, false, 8, DEPTH, 16, false> R;
    constexpr int D = R::D;
    extern __shared__ __attribute__((aligned(16))) u32 dyn[];
    const u32 wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, W = blockDim.x >> 6;
    const u32 fbs = ff / 128, cbs = hidden / 128, U = 4 * fbs;   // U: units a column block
    u32 share;
    const u32 item = xpf_place(parts, share);
    const XpfItem it = xpf_item(offs, items, item, ne, sh_addr != nullptr, 16 * ntl);
    if (it.n == 0) return;
    const u8* down = (const u8*) uniform_u64(it.e < ne ? eaddr[2ull * ne + it.e] : sh_addr[2]);
    const u32 cb0 = share * W + wave, stride = parts * W;        // the wave's column blocks: cb0, cb0 + stride, ..
    u16* xrows = (u16*) dyn;
    float* fac = (float*) (dyn + ntl * fbs * 1024);
    u16* scales = (u16*) (fac + ntl * fbs * 16) + wave * XPF_DOWN_BLOCKS * 128;   // of the wave's column blocks
    u32* wb = dyn + ntl * fbs * 1040 + W * XPF_DOWN_BLOCKS * 64 + wave * (D * R::UW);
    const u32 blocks = cb0 < cbs ? (cbs - cb0 + stride - 1) / stride : 0u, total = blocks * U;
    R ring;
    ring.init(down + 2 * (u64) ff + 2 * (u64) hidden + 4 + (u64) (cb0 < cbs ? cb0 : 0) * 8 * (4 * R::TW), (hidden / 16) * (4 * R::TW), U, __builtin_amdgcn_readfirstlane(lds_offset(wb)), lane);
    xpf_tiles<XPF_DOWN_NT>(it.tiles, [&](auto n) {
        constexpr int NT = decltype(n)::value < XPF_DOWN_NT ? decltype(n)::value : XPF_DOWN_NT;
        u32 pair[NT];
#pragma unroll
        for (int T = 0; T < NT; T++) pair[T] = list[it.first + min(16 * T + (lane & 15), it.n - 1)];
#pragma unroll
        for (int T = 0; T < NT; T++) load_landed(pair[T]);
        for (u32 i = wave; i < it.tiles * fbs * 4; i += W) lds_load<16>((const u8*) (rows + (u64) it.base * fbs * XPF_ROWS_U16) + i * 1024 + lane * 16, lds_offset(xrows) + i * 1024);
        for (u32 i = wave; 64 * i < it.tiles * fbs * 16; i += W)
            if (64 * i + lane < it.tiles * fbs * 16) lds_load<4>(inv + it.base * fbs * 16 + 64 * i + lane, lds_offset(fac) + 256 * i);
        for (u32 i = 0; i < blocks; i++) lds_load<4>(down + 2 * (u64) ff + 256 * (cb0 + i * stride) + 4 * lane, lds_offset(scales) + 256 * i);
        // the unit after the last one requested: where it lies
        u32 ahead = 0, unit = 0;
        auto request = [&](u32 slot) {
            ring.issue(unit, slot, lane);
            ahead++;
            if (++unit == U) {
                unit = 0;
                ring.row0 += (u64) stride * 8 * (4 * R::TW);
            }
        };
        if (total) {
#pragma unroll
            for (int d = 0; d < D; d++)
                if ((u32) d < total) request(d);
            if (total >= (u32) D) wait_vm<D * R::NI>();
            else wait_vm<0>();
        } else wait_vm<0>();
        lds_barrier();
        // blocks that xpf_chain drops: zeros in their place
        if (threadIdx.x < 16 * it.tiles) {
            const u32 T = threadIdx.x / 16, t = threadIdx.x % 16;
            xpf_chain(fac + T * fbs * 16 + t, fbs, [&](u32 b) {
                for (u32 i = 0; i < 16; i++) *(u32x4*) (xrows + (T * fbs + b) * XPF_ROWS_U16 + (16 * i + t) * 8) = u32x4{0, 0, 0, 0};
            });
        }
        lds_barrier();
        if (!total) return;
        typedef XpfStep<K, 8, NT> Step;
        const u32 tstep = fbs * XPF_ROWS_U16;
        Step s0, s1;
        u32x4 xv[NT], xn[NT];
        f32x4 acc[NT][8];
        auto reset = [&] {
#pragma unroll
            for (int T = 0; T < NT; T++)
#pragma unroll
                for (int c = 0; c < 8; c++) acc[T][c] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        };
        auto factor = [&](int T, u32 b) { return fac[(min((u32) T, it.tiles - 1) * fbs + b) * 16 + (lane & 15)]; };   // what undoes the power of two
        reset();
        if (total >= (u32) D) wait_vm<(D - 1) * R::NI>();
        s0.read(wb, 0, lane);
        Step::rows(xv, xrows + lane * 8, tstep);
        u32 slot = 0, u = 0, done = 0;   // done: column blocks finished
#pragma unroll 1
        for (u32 g = 0; g < total; g++) {
            s1.read(wb + slot * R::UW, 1, lane);
            __builtin_amdgcn_sched_barrier(0);
            if ((u & 3) == 0 && u > 0) {
                // another 128-block of the inputs: its tokens' powers of two mostly are the ones before
#pragma unroll
                for (int T = 0; T < NT; T++) {
                    const float r = factor(T, u / 4 - 1) / factor(T, u / 4);   // a power of two
                    if (__builtin_amdgcn_ballot_w64(r != 1.0f)) {
#pragma unroll
                        for (int c = 0; c < 8; c++) acc[T][c] *= r;
                    }
                }
            }
            s0.template products<0>(xv, acc, lane);
            __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0): the unit's words are in registers, its slot can take the unit D further on
            if (ahead < total) request(slot);
            slot = slot + 1 == (u32) D ? 0u : slot + 1;
            const u32 un = u + 1 == U ? 0u : u + 1;
            if (g + 1 < total) {
                // behind the next unit: D - 1 units, but for the stream's end, and the stores of a finished block, which count too
                if (g + 1 + D > total) wait_vm<0>();
                else if (done > 0 && u + 1 < (u32) D) wait_vm<(D - 1) * R::NI + 8 * (NT <= 2 ? NT : NT - 1)>();
                else wait_vm<(D - 1) * R::NI>();
                s0.read(wb + slot * R::UW, 0, lane);
                Step::rows(xn, xrows + un * 512 + lane * 8, tstep);
                __builtin_amdgcn_sched_barrier(0);
            }
            s1.template products<4>(xv, acc, lane);
            u = un;
            if (u == 0) {
#pragma unroll
                for (int T = 0; T < NT; T++) {
                    const float f = factor(T, fbs - 1);
#pragma unroll
                    for (int c = 0; c < 8; c++) acc[T][c] *= f;
                    xpf_transform(acc[T]);
                    if (16 * T + (lane & 15) < it.n) {
                        float* o = eo + (u64) pair[T] * hidden + (cb0 + done * stride) * 128;
#pragma unroll
                        for (int c = 0; c < 8; c++) {
                            const u16x4 s4 = *(const u16x4*) (scales + done * 128 + xpf_out_col(c, lane));
                            f32x4 v;
#pragma unroll
                            for (int q = 0; q < 4; q++) v[q] = acc[T][c][q] * (f16_to_f32(s4[q]) * 0.08838835f);
                            *(f32x4*) (o + xpf_out_col(c, lane)) = v;
                        }
                    }
                }
                reset();
                done++;
            }
#pragma unroll
            for (int T = 0; T < NT; T++) xv[T] = xn[T];
        }
    });
}

#define EXL3_PREFILL_ENTRIES(K) \
    extern "C" __global__ void __launch_bounds__(512, 2) prefill_gate_up_exl3_##K(const u64* eaddr, const u64* sh_addr, const u32* offs, const u32* items, const u16* rows, const float* inv, u16* rows2, \
                                                                                  float* inv2, u32 ne, u32 hidden, u32 ff, u32 tok) { \
        prefill_gate_up_exl3_kernel<K, 2>(eaddr, sh_addr, offs, items, rows, inv, rows2, inv2, ne, hidden, ff, tok); \
    } \
    extern "C" __global__ void __launch_bounds__(512, 4) prefill_gate_up_n_exl3_##K(const u64* eaddr, const u64* sh_addr, const u32* offs, const u32* items, const u16* rows, const float* inv, u16* rows2, \
                                                                                    float* inv2, u32 ne, u32 hidden, u32 ff, u32 tok) { \
        prefill_gate_up_exl3_kernel<K, 1>(eaddr, sh_addr, offs, items, rows, inv, rows2, inv2, ne, hidden, ff, tok); \
    } \
    extern "C" __global__ void __launch_bounds__(512, 2) prefill_down_exl3_##K(const u64* eaddr, const u64* sh_addr, const u32* offs, const u32* list, const u32* items, const u16* rows, const float* inv, \
                                                                               float* eo, u32 ne, u32 hidden, u32 ff, u32 ntl, u32 parts) { \
        prefill_down_exl3_kernel<K, XPF_RING(K)>(eaddr, sh_addr, offs, list, items, rows, inv, eo, ne, hidden, ff, ntl, parts); \
    } \
    extern "C" __global__ void __launch_bounds__(256, 2) prefill_down_n_exl3_##K(const u64* eaddr, const u64* sh_addr, const u32* offs, const u32* list, const u32* items, const u16* rows, const float* inv, \
                                                                                 float* eo, u32 ne, u32 hidden, u32 ff, u32 ntl, u32 parts) { \
        prefill_down_exl3_kernel<K, XPF_RING_DOWN_N(K)>(eaddr, sh_addr, offs, list, items, rows, inv, eo, ne, hidden, ff, ntl, parts); \
    }
EXL3_PREFILL_ENTRIES(1)
EXL3_PREFILL_ENTRIES(2)
EXL3_PREFILL_ENTRIES(3)
EXL3_PREFILL_ENTRIES(4)
EXL3_PREFILL_ENTRIES(5)
EXL3_PREFILL_ENTRIES(6)
EXL3_PREFILL_ENTRIES(7)
EXL3_PREFILL_ENTRIES(8)

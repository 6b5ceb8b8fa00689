// The prefill chunk of one MoE layer on int8 activations: tokens grouped by expert, IQ3_S weights decoded to whole numbers in f16, f16 MFMA
// tiles (v_mfma_f32_16x16x32_f16: 16 weight rows x 16 tokens x one 32-weight sub-block), a sub-block's exact sums scaled by the
// activations' scale in f32, SwiGLU, H re-quantized per 32, down into pair rows.
//
// Arithmetic follows the reference's CPU statement of the int8-activation expert (crates/shadowzero-model/src/cpu_expert.rs:99-110,
// 144-155, 217, 298-339 and cpu_expert_avx512.rs:25-42) with activation blocks of 32: d_x = amax / 127,
// q = clamp(round-half-away(v / d_x)); weights grid * sign with s_w = d (1 + 2 scale) per 32.  Codes (up to 127) and
// grid * sign * (1 + 2 scale) (up to 465) are whole numbers, exact in f16, and 32 products of theirs stay below 2^24: the matrix
// instruction's f32 sum of a sub-block is exact.  A row's product is, per 256 weights, d times the sum over the sub-blocks of
// d_x * sum, both steps fused multiply-adds in f32 (the CPU statement adds (s_w * d_x) * sum sub-block by sub-block: other
// roundings of the last bits).  Codes are multiplied by 2^-6 and weights by 2^-14, exactly, and d by 2^20: sums of the largest finite
// activations then stay finite until d is in.  The launch structure is the native fused path's (native/fused/shadowzero_fused.cu:5-9: quantize,
// group, experts), re-made for wave64 MFMA.
//
// Why f16 and not the int8 instruction: int8 weights leave the scale 1 + 2 s out, and every sum then takes a conversion, a product of
// scales and a multiply-add, 12 vector instructions a tile and sub-block where this form takes 4 (and a matrix instruction of
// the same length).
//
// MFMA operand layout: A (weight rows x k) lane l holds row l % 16, k = 8 (l / 16) .. +8; B (k x tokens) lane l holds token l % 16, the
// same k; C lane l holds token l % 16, weight rows 4 (l / 16) + r in element r.

//
// The ahead-of-time build has the matrix instructions write to ordinary vector registers: every tile's 4 sums a lane are
// scaled at once, and out of the accumulation registers each would first cost a move.
// hipcc: -mllvm -amdgpu-mfma-vgpr-form=1

typedef u32 u32x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ u32 f16_pair(float a, float b) { return __builtin_bit_cast(u32, f16x2{(_Float16) a, (_Float16) b}); }

// q[i] = clamp(round(x[i] / d)), d[b] = amax / 127 over each 32 values (cpu_expert_avx512.rs:25-42); h (where not null): the codes
// again, times 2^-6, as f16.  One thread a block of 32.
__device__ __forceinline__ void quant_block_q8(const float* x, u64 b, i8* q, float* d, u16* h) {
    const f32x4* p = (const f32x4*) (x + b * 32);
    float v[32];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const f32x4 t = p[i];
        v[4 * i] = t.x;
        v[4 * i + 1] = t.y;
        v[4 * i + 2] = t.z;
        v[4 * i + 3] = t.w;
    }
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < 32; i++) amax = fmaxf(amax, fabsf(v[i]));
    const float dd = amax / 127.0f;
    const float id = dd > 0.0f ? 1.0f / dd : 0.0f;
    u32 w[8];
#pragma unroll
    for (int i = 0; i < 32; i++) v[i] = fminf(127.0f, fmaxf(-127.0f, roundf(v[i] * id)));
#pragma unroll
    for (int i = 0; i < 8; i++) {
        u32 pack = 0;
#pragma unroll
        for (int k = 0; k < 4; k++) pack |= ((u32) (int) v[4 * i + k] & 0xffu) << (8 * k);
        w[i] = pack;
    }
    u32x4* o = (u32x4*) (q + b * 32);
    o[0] = u32x4{w[0], w[1], w[2], w[3]};
    o[1] = u32x4{w[4], w[5], w[6], w[7]};
    if (h) {
        u32x4* oh = (u32x4*) (h + b * 32);
#pragma unroll
        for (int i = 0; i < 32; i++) v[i] *= 0x1p-6f;
#pragma unroll
        for (int i = 0; i < 4; i++)
            oh[i] = u32x4{f16_pair(v[8 * i], v[8 * i + 1]), f16_pair(v[8 * i + 2], v[8 * i + 3]), f16_pair(v[8 * i + 4], v[8 * i + 5]), f16_pair(v[8 * i + 6], v[8 * i + 7])};
    }
    d[b] = dd;
}

// grid = ceil(n / 32 / 256), block 256.
extern "C" __global__ void __launch_bounds__(256) quant_act_q8(const float* x, u64 n, i8* q, float* d) {
    const u64 b = (u64) blockIdx.x * 256 + threadIdx.x;
    if (b < n / 32) quant_block_q8(x, b, q, d, nullptr);
}

// The two things a chunk needs before its tokens can be grouped, in one launch (they do not depend on each other): the
// routing of its m tokens (workgroups [0, ceil(m / 4)): a wave a token, as route_topk_rows) and the quantization of its
// activations (the workgroups after them, as quant_act_q8).  grid = ceil(m / 4) + ceil(n / 32 / 256), block 256.
extern "C" __global__ void __launch_bounds__(256) prefill_front(const float* x, u64 n, i8* q, float* d, u16* h, const float* logits, u32* tidx, float* weights, u32* cnt,
                                                                u32 ne, u32 k, u32 m) {
    __shared__ double exs[4][512];
    __shared__ u32 tops[4][16];
    const u32 nr = (m + 3) / 4;
    if (blockIdx.x >= nr) {
        const u64 b = (u64) (blockIdx.x - nr) * 256 + threadIdx.x;
        if (b < n / 32) quant_block_q8(x, b, q, d, h);
        return;
    }
    const u32 lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const u32 j = blockIdx.x * 4 + w;
    if (j >= m) return;
    route_ids(logits + (u64) j * ne, ne, k, lane, exs[w], tops[w]);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    u32 count;
    const float wt = route_weights_chosen(logits + (u64) j * ne, ne, k, lane, tops[w], &count);
    if (lane < k) {
        tidx[(u64) j * k + lane] = tops[w][lane];
        weights[(u64) j * k + lane] = wt;
    }
    if (lane == 0) cnt[j] = count;
}

#define PF_TOK 64      // tokens of one work item: PF_TOK / 16 MFMA tiles of 16
#define PF_TILES (PF_TOK / 16)

// Groups the chunk's (token, rank) pairs by expert: offs[e] .. offs[e + 1] are the positions in list[] of expert e's pairs
// (pair = token * k + rank; the shared expert, index ne, takes the pairs npairs + token when nshared = tokens).  The order of an expert's pairs in list[] is
// arbitrary; every pair owns its output rows, so the results do not depend on it.  items[0] = the number of work items, items[1 + 2 i], items[2 + 2 i] =
// (expert, first position) of item i: every run of up to unit_gu pairs of an expert is one item of the gate/up kernel (at most
// ne + 1 + rows / unit_gu of them); items_d likewise with runs of up to unit_d pairs, for the down kernel.  The longest items come
// first, so that the launches end on short ones, and all ahead of the workgroups launched for the rest of the bound (int8 chunk of 512
// tokens: 239 -> 226 us with the order alone).  items_d may be null.
// Up to 4096 pairs one workgroup does it all (prefill_group).  For more (prefill_group_many) every workgroup counts all pairs; the first then writes offs and the
// items, the others list `share` pairs each, whose places in an expert's run the count of the pairs ahead of them tells: nothing passes between workgroups.
// Bound by the counting, lots of loads and the LDS additions of popular experts.  40960 pairs 29.5 -> 16.8 us, 5120 9.6 -> 6.5, where one
// workgroup did it all; 450 pairs 4.6 either way, which the common form would make 4.9.
template <bool many>
__device__ __forceinline__ void prefill_group_body(const u32* tidx, u32 tokens, u32 k, u32 ne, u32 nshared, u32* offs, u32* list, u32* items, u32* items_d, u32 unit_gu, u32 unit_d, u32 share) {
    __shared__ u32 s_cnt[513], s_off[514], s_ahead[513], s_full[2][513], s_class[2][9];
    const u32 tid = threadIdx.x, npairs = tokens * k, nexp = ne + 1;
    const u32 b = many ? blockIdx.x : 0u, from = !many ? 0u : b ? min((b - 1) * share, npairs) : npairs, to = many ? min(from + share, npairs) : npairs;   // the pairs it lists
    for (u32 i = tid; i < nexp; i += 1024) {
        s_cnt[i] = 0;
        s_ahead[i] = 0;
    }
    if (tid < 18) s_class[tid / 9][tid % 9] = 0;
    __syncthreads();
    // 32 pairs of a thread in flight at a time: the loads' round trips are what this launch is made of; as many as there are where those are few
    // (1200 pairs 8.0 us with 32, 5.0 with four)
    auto lot = [&](auto depth, u32 p0, u32 end, auto use) {
        constexpr int N = sizeof(depth);
        u32 e[N];
#pragma unroll
        for (int q = 0; q < N; q++) e[q] = tidx[min(p0 + 1024 * q, npairs - 1)];
#pragma unroll
        for (int q = 0; q < N; q++)
            if (p0 + 1024 * q < end && e[q] < ne) use(p0 + 1024 * q, e[q]);
    };
    struct Many {
        u8 of[32];
    };
    auto few = [&](u32 p0, u32 end, auto use) {
        if (!many && npairs <= 1024) {
            if (tid < npairs) lot(u8(), tid, npairs, use);
        } else
            for (; p0 < end; p0 += 4 * 1024) lot(u32(), p0, end, use);
    };
    if (many)
        for (u32 p0 = tid; p0 < npairs; p0 += 32 * 1024) lot(Many(), p0, npairs, [&](u32 p, u32 e) { atomicAdd(p < from ? &s_ahead[e] : &s_cnt[e], 1u); });
    else few(tid, npairs, [&](u32, u32 e) { atomicAdd(&s_cnt[e], 1u); });
    if (tid == 0) s_cnt[ne] = nshared;
    __syncthreads();
    if (from) {   // (uniform)
        for (u32 i = tid; i < nexp; i += 1024) s_cnt[i] += s_ahead[i];
        __syncthreads();
    }
    // three running sums over the experts, each by a wave of its own: lane L takes the experts [9 L, 9 L + 9) (ne <= 512), the
    // lanes' totals are scanned across the wave, and every lane writes its experts' starts: of the pairs, of the full items of
    // either list
    {
        const u32 w = tid >> 6, lane = tid & 63;
        if (w < 3) {
            const u32 unit = w == 0 ? 1u : w == 1 ? unit_gu : unit_d;
            u32 v[9], sum = 0;
#pragma unroll
            for (int q = 0; q < 9; q++) {
                const u32 i = 9 * lane + q;
                v[q] = i < nexp ? s_cnt[i] / unit : 0u;
                sum += v[q];
            }
            u32 incl = sum;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const u32 up = __shfl_up(incl, o, SZ_WAVE);
                if (lane >= (u32) o) incl += up;
            }
            u32 run = incl - sum;
            u32* dst = w == 0 ? s_off : s_full[w - 1];
#pragma unroll
            for (int q = 0; q < 9; q++) {
                const u32 i = 9 * lane + q;
                if (i < nexp) dst[i] = run;
                run += v[q];
            }
            if (lane == 63) {
                if (w == 0) s_off[nexp] = incl;
                else s_class[w - 1][0] = incl;
            }
        } else {
            // the items that are not full, by the number of their tiles of 16 pairs
            for (u32 i = tid - 192; b == 0 && i < (items_d ? 2 : 1) * nexp; i += 1024 - 192) {
                const u32 l = i >= nexp ? 1u : 0u, unit = l ? unit_d : unit_gu, rest = s_cnt[i - l * nexp] % unit;
                if (rest) atomicAdd(&s_class[l][1 + min((unit - rest) / 16, 7u)], 1u);
            }
        }
    }
    __syncthreads();
    auto lists = [&] {
        few(from + tid, to, [&](u32 p, u32 e) { list[s_off[e] + atomicAdd(&s_ahead[e], 1u)] = p; });
        for (u32 j = b * 1024 + tid; j < nshared; j += (many ? gridDim.x : 1u) * 1024) list[s_off[ne] + j] = npairs + j;
    };
    if (b) return lists();
    if (tid < (items_d ? 2u : 1u)) {   // where the full ones end and each class begins, the longest first
        u32 run = 0;
        for (u32 c = 0; c < 9; c++) {
            const u32 n = s_class[tid][c];
            s_class[tid][c] = run;
            run += n;
        }
        (tid ? items_d : items)[0] = run;
    }
    __syncthreads();
    for (u32 i = tid; i < (items_d ? 2 : 1) * nexp; i += 1024) {
        const u32 l = i >= nexp ? 1u : 0u, e = i - l * nexp, unit = l ? unit_d : unit_gu, n = s_cnt[e], rest = n % unit;
        u32* to = l ? items_d : items;
        u32 at = s_full[l][e], t0 = 0;
        for (; t0 + unit <= n; t0 += unit, at++) {
            to[1 + 2 * at] = e;
            to[2 + 2 * at] = t0;
        }
        if (rest) {
            at = atomicAdd(&s_class[l][1 + min((unit - rest) / 16, 7u)], 1u);
            to[1 + 2 * at] = e;
            to[2 + 2 * at] = t0;
        }
    }
    for (u32 i = tid; i <= nexp; i += 1024) offs[i] = s_off[i];
    lists();
}
// At most 4096 pairs.  grid 1, block 1024; ne <= 512.
extern "C" __global__ void __launch_bounds__(1024) prefill_group(const u32* tidx, u32 tokens, u32 k, u32 ne, u32 nshared, u32* offs, u32* list,
                                                                 u32* items, u32* items_d, u32 unit_gu, u32 unit_d) {
    prefill_group_body<false>(tidx, tokens, k, ne, nshared, offs, list, items, items_d, unit_gu, unit_d, 0);
}
// grid = 1 + ceil(pairs / share), block 1024; ne <= 512.
extern "C" __global__ void __launch_bounds__(1024) prefill_group_many(const u32* tidx, u32 tokens, u32 k, u32 ne, u32 nshared, u32* offs, u32* list,
                                                                      u32* items, u32* items_d, u32 unit_gu, u32 unit_d, u32 share) {
    prefill_group_body<true>(tidx, tokens, k, ne, nshared, offs, list, items, items_d, unit_gu, unit_d, share);
}

// A workgroup's LDS.  The grid comes first: its address fits the look-ups' constant offset.
#define PF_STAGE 73728
struct PfLds {
    u32x2 grid[512];   // the codebook grid, a weight's magnitude as f16
    u8 stage[PF_STAGE];
    u32 rows[PF_TOK], pairs[PF_TOK];
    float strip[8][16];
};

// Fills the table; every thread of the workgroup (512) calls it, and a barrier must follow before it is read.
__device__ __forceinline__ void pf_tables(u32x2* grid, u32 tid) {
    const u32 g = IQ3S_GRID[tid];
    grid[tid] = u32x2{f16_pair((float) (g & 0xff), (float) ((g >> 8) & 0xff)), f16_pair((float) ((g >> 16) & 0xff), (float) (g >> 24))};
}

// Eight consecutive weights (k = 8 kq .. 8 kq + 7 of sub-block g) of one IQ3_S block at `blk` (LDS, 2-byte aligned) as f16: grid * sign
// (cpu_expert.rs:99-110) * (1 + 2 scale), `scale` holding the last factor twice; qh: bits 0 and 1 the ninth bits of the two grid indexes.  The two
// signs of a pair are moved to the sign bits of its halves by one multiplication (the two copies of the sign byte that it
// makes do not overlap).
__device__ __forceinline__ f16x8 iq3s_f16x8(const u32x2* grid, const u8* blk, u32 g, u32 kq, u32 qh, f16x2 scale) {
    const u32 qs = *(const u16*) (blk + 2 + 8 * g + 2 * kq);   // the low bytes of the two 4-weight groups' grid indexes
    const u32 signs = blk[74 + 4 * g + kq];
    u32 at0 = (qs & 0xff) << 3 | ((qh << 11) & 0x800u), at1 = (qs >> 8) << 3 | ((qh << 10) & 0x800u);
    asm("" : "+v"(at0), "+v"(at1));   // bytes into the table, whose own address then is the loads' constant offset
    const u32x2 g0 = *(const u32x2*) ((const u8*) grid + at0), g1 = *(const u32x2*) ((const u8*) grid + at1);
    auto pair = [&](u32 of, u32 spread) {
        return __builtin_bit_cast(u32, __builtin_bit_cast(f16x2, of) * __builtin_bit_cast(f16x2, ((signs * spread) & 0x80008000u) ^ __builtin_bit_cast(u32, scale)));
    };
    return __builtin_bit_cast(f16x8, u32x4{pair(g0.x, 0x40008000u), pair(g0.y, 0x10002000u), pair(g1.x, 0x04000800u), pair(g1.y, 0x01000200u)});
}

// (1 + 2 s) 2^-14 twice, s the four bits from `bit` on.
__device__ __forceinline__ f16x2 iq3s_scale_pair(u32 sc, u32 bit) {
    const f16x2 v = __builtin_bit_cast(f16x2, __builtin_amdgcn_ubfe(sc, bit, 4) * 0x20002u + 0x2c012c01u);   // 2^-4 + (1 + 2 s) 2^-14
    return v - f16x2{(_Float16) 0x1p-4f, (_Float16) 0x1p-4f};
}

#define PF_WB 7168             // 64 rows' blocks of one matrix in LDS: 28 words a row
#define PF_WS 112              // bytes between rows there

__device__ __forceinline__ u64 uniform_u64(u64 v) {
    return ((u64) (u32) __builtin_amdgcn_readfirstlane((u32) (v >> 32)) << 32) | (u32) __builtin_amdgcn_readfirstlane((u32) v);
}
// lds_load_at's 4-byte form
__device__ __forceinline__ void pf_load4_at(u64 base, u32 off, u32 lds) {
    u32 keep;
    lds = __builtin_amdgcn_readfirstlane(lds);
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %1, %3\n\ts_mov_b32 m0, %0" : "=&s"(keep) : "v"(off), "s"(lds), "s"(base) : "memory");
}

// The same block (256 weights) of 64 consecutive rows of a row-major IQ3_S matrix: 28 words a row.  Blocks are only 2-byte
// aligned: a row's words start at the word that holds the block's first byte, and the block begins pf_shift (0 or 2) bytes
// into its slot.  The words of a row never leave the matrix: its first block starts on a word and its last one ends on one (a
// row is a multiple of 4 bytes, or rows come in even numbers).  at = the first of the 64 rows' block, rb = bytes a row.
__device__ __forceinline__ u32 pf_shift(u64 at, u32 rb, u32 row) { return ((u32) at + row * rb) & 2; }
struct PfRows {
    u32 off[4];   // the lane's word in the wave's load instructions, of 28: 64 rows x 28 words
    static __device__ __forceinline__ u32 place(u32 it, u32 wave) { return it < 3 ? wave + 8 * it : 24 + (wave & 3); }
    __device__ __forceinline__ void init(u32 rb, u32 wave, u32 lane) {
#pragma unroll
        for (u32 it = 0; it < 4; it++) {
            const u32 i = place(it, wave) * 64 + lane;
            off[it] = i / 28 * rb + i % 28 * 4;
        }
    }
    // the wave's share of the instructions, 3 or 4 of 8 waves' 28; with `mirrored` 4 or 3: of two calls 7
    template <bool mirrored>
    __device__ __forceinline__ void issue(u64 at, u32 lds_w, u32 wave) const {
#pragma unroll
        for (u32 it = 0; it < 4; it++)
            if (it < 3 || (mirrored ? wave >= 4 : wave < 4))   // (wave-uniform)
                pf_load4_at(at & ~3ull, (off[it] + ((u32) at & 3)) & ~3u, lds_w + place(it, wave) * 256);
    }
};

// Half a block's products (128 weights, 4 sub-blocks) with the first T token tiles: acc += d_x * a sub-block's exact sum, in sub-block order.
// xs, ds: the half's activations and their scales ([sub-block][64 tokens]); blk: the lane's row's block in LDS.
template <int T>
__device__ __forceinline__ void pf_products(f32x4 (&acc)[T], const u32x2* grid, const u8* xs, const float* ds, const u8* blk, u32 half, u32 n, u32 kq) {
    f16x8 w[4];
    const u32 qh = ((u32) *(const u16*) (blk + 66 + 4 * half) | (u32) *(const u16*) (blk + 68 + 4 * half) << 16) >> (2 * kq);
#pragma unroll
    for (int j = 0; j < 4; j++) w[j] = iq3s_f16x8(grid, blk, 4 * half + j, kq, qh >> (8 * j), iq3s_scale_pair(blk[106 + 2 * half + j / 2], 4 * (j % 2)));
    __builtin_amdgcn_sched_barrier(0);
    // a step is a tile and sub-block: its operands are read a step ahead, its sums scaled while the next one's are made
    auto read = [&](int step, f16x8& x, float& dx) {
        const u32 a = step / 4, g = step % 4;
        x = *(const f16x8*) (xs + (16 * a + n) * 256 + ((4 * g + kq) ^ n) * 16);
        dx = ds[g * PF_TOK + 16 * a + n];
    };
    f16x8 x[2];
    float dx[3];
    f32x4 c[2];
    read(0, x[0], dx[0]);
#pragma unroll
    for (int step = 0; step <= 4 * T; step++) {
        if (step + 1 < 4 * T) read(step + 1, x[(step + 1) % 2], dx[(step + 1) % 3]);
        if (step < 4 * T) c[step % 2] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[step % 4], x[step % 2], f32x4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
        if (step > 0) {
            f32x4& sum = acc[(step - 1) / 4];
#pragma unroll
            for (int r = 0; r < 4; r++) sum[r] = __builtin_fmaf(dx[(step - 1) % 3], c[(step - 1) % 2][r], sum[r]);
            asm volatile("" : "+v"(sum));   // here, and not where the sums are next used: the products' registers are needed
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// A block is complete: total += 2^20 d * acc, d the f16 scale of the block of each of the lane's four rows, which the lanes of the rows hand over
// through the wave's own strip of LDS (a wave's LDS operations are in order).
template <int T>
__device__ __forceinline__ void pf_fold(f32x4 (&total)[T], f32x4 (&acc)[T], const u8* blk, float* strip, u32 n, u32 kq) {
    if (kq == 0) strip[n] = f16_to_f32(*(const u16*) blk) * 0x1p20f;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const f32x4 d = *(const f32x4*) (strip + 4 * kq);
#pragma unroll
    for (int a = 0; a < T; a++) {
#pragma unroll
        for (int r = 0; r < 4; r++) total[a][r] = __builtin_fmaf(d[r], acc[a][r], total[a][r]);
        acc[a] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
}

// The products of a workgroup of 8 waves: T tiles of an item's tokens with 128 rows, waves 0 .. 3 the 64 that begin at w0, waves 4 .. 7 the
// 64 at w1, 16 each; `blocks` IQ3_S blocks of every row, nc of them (the whole row) for one lot of 128 rows, whose sums go to
// finish(lot, total), then nc of the rows `lot` bytes further on.  x, d: the codes and scales of `cols` inputs a row, s_rows (LDS): the
// row of every token.
//
// Blocks and activations come into LDS by global-to-LDS loads, a wave's load instruction filling 64 consecutive slots from 64 addresses of
// its choosing: the layout is made by choosing the addresses.  Token t's 16-byte column c lands at slot c ^ (t & 15) of its row, so
// that the 16 tokens of an MFMA tile read the same column from 16 different bank groups.  For one or two tiles a whole block of
// the rows with its activations is a stage, three or two of them in flight (an item of one tile has little to multiply while it
// waits); for three and four the activations come a half block at a time, one ahead, the rows a block ahead.  Two workgroups a
// compute unit by the stage's LDS.
//
// What bounds it: the decode, about 25 vector instructions for a lane's 8 weights, for every item of an expert again, then LDS, busy half the time
// (the grid look-ups' bank conflicts), and the waits of items of one tile.  512 tokens through 512 experts of 2048 x 512, top-10, router
// with Zipf's preferences: gate and up 138 -> 111 us, down 82 -> 61, the chunk 229 -> 169; 4096 tokens and the shared expert 1092 ->
// 843; 700 through 60 of 4096 x 1536, top-4, 582 -> 418.  Tried: 16 rows of either matrix and half the sub-blocks a wave, which reads
// the activations half as often (gate and up 112, down 78).
template <int T, class F>
__device__ __forceinline__ void pf_stream(PfLds& lds, u64 w0, u64 w1, u64 lot, u32 rb, u32 nc, u32 blocks, const u16* __restrict__ x, const float* __restrict__ d, const u32* s_rows, u32 cols,
                                          u32 wave, u32 lane, F&& finish) {
    constexpr u32 XB = T * 4096;   // half a block's activations: [16 T tokens][16 columns of 8 codes]
    u8* stage = lds.stage;
    float* strip = lds.strip[wave];
    const u32 n = lane & 15, kq = lane >> 4, lrow = (wave & 3) * 16 + n, mine = wave >> 2, lds0 = __builtin_amdgcn_readfirstlane(lds_offset(stage));
    PfRows rows;
    rows.init(rb, wave, lane);
    auto input = [&](u32 j) {   // the lane's part of an instruction of 4 tokens
        const u32 t = 4 * j + (lane >> 4);
        return x + (u64) s_rows[t] * cols + 8 * ((lane & 15) ^ (t & 15));
    };
    f32x4 acc[T], total[T];
#pragma unroll
    for (int a = 0; a < T; a++) acc[a] = total[a] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    u32 ahead = 0;             // blocks asked for; of these in the current lot, and its number
    u32 ac = 0, ab = 0;
    u64 a0 = w0, a1 = w1;
    auto next = [&] {
        ahead++;
        a0 += 110;
        a1 += 110;
        if (++ac == nc) {
            ac = 0;
            ab++;
            a0 = w0 + ab * lot;
            a1 = w1 + ab * lot;
        }
    };
    u64 at = mine ? w1 : w0;   // the wave's block
    u32 c = 0, done = 0;
    auto fold = [&](const u8* blk) {
        pf_fold<T>(total, acc, blk, strip, n, kq);
        at += 110;
        if (++c == nc) {
            finish(done, total);
#pragma unroll
            for (int a = 0; a < T; a++) total[a] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            c = 0;
            done++;
            at = (mine ? w1 : w0) + done * lot;
        }
    };
    if constexpr (T <= 2) {
        constexpr u32 D = T == 1 ? 3 : 2, WO = 2 * XB, DO = WO + 2 * PF_WB, SB = DO + 2048, A = 7 + T + 1;   // A: a wave's loads a stage
        static_assert(D * SB <= PF_STAGE, "the stages' LDS");
        const u16* xp = input(T == 1 ? wave & 3 : wave);
        const float* dp = d + (u64) s_rows[lane] * (cols / 32) + wave;
        auto request = [&](u32 slot) {
            const u32 to = lds0 + slot * SB;
            if constexpr (T == 1) lds_load<16>(xp + ac * 256 + (wave >> 2) * 128, to + wave * 1024);
            else {
                lds_load<16>(xp + ac * 256, to + wave * 1024);
                lds_load<16>(xp + ac * 256 + 128, to + XB + wave * 1024);
            }
            rows.issue<false>(a0, to + WO, wave);
            rows.issue<true>(a1, to + WO + PF_WB, wave);
            lds_load<4>(dp + ac * 8, to + DO + wave * 256);   // a sub-block's 64
            next();
        };
#pragma unroll
        for (u32 i = 0; i + 1 < D; i++)
            if (i < blocks) request(i);
        u32 slot = 0;
#pragma unroll 1
        for (u32 b = 0; b < blocks; b++) {
            if (D == 3 && ahead > b + 1) wait_vm<(D - 2) * A>();
            else wait_vm<0>();
            __syncthreads();   // block b is in LDS, from every wave; the products of block b - 1 are done, so its slot is free
            const u8* s = stage + slot * SB;
            if (ahead < blocks) request(slot == 0 ? D - 1 : slot - 1);
            slot = slot + 1 == D ? 0u : slot + 1;
            const u8* blk = s + WO + mine * PF_WB + lrow * PF_WS + pf_shift(at, rb, lrow);
            pf_products<T>(acc, lds.grid, s, (const float*) (s + DO), blk, 0, n, kq);
            pf_products<T>(acc, lds.grid, s + XB, (const float*) (s + DO + 1024), blk, 1, n, kq);
            fold(blk);
        }
    } else {
        constexpr u32 WO = 2 * XB, DO = WO + 4 * PF_WB;
        static_assert(DO + 2048 <= PF_STAGE, "the stages' LDS");
        const u16* xp[2] = {input(wave), input(wave + 8)};
        const float* dp = d + (u64) s_rows[lane] * (cols / 32) + (wave & 3);
        auto inputs = [&](u32 u, u32 slot) {   // half u of a row's inputs
            lds_load<16>(xp[0] + u * 128, lds0 + slot * XB + wave * 1024);
            if (T == 4 || wave < 4) lds_load<16>(xp[1] + u * 128, lds0 + slot * XB + (wave + 8) * 1024);
            if (wave < 4) lds_load<4>(dp + u * 4, lds0 + DO + slot * 1024 + wave * 256);
        };
        rows.issue<false>(a0, lds0 + WO, wave);
        rows.issue<true>(a1, lds0 + WO + PF_WB, wave);
        next();
        inputs(0, 0);
#pragma unroll 1
        for (u32 b = 0; b < blocks; b++) {
            const u8* blk = stage + WO + ((b & 1) * 2 + mine) * PF_WB + lrow * PF_WS + pf_shift(at, rb, lrow);
            const u32 to = lds0 + WO + ((b + 1) & 1) * 2 * PF_WB;
            wait_vm<0>();
            __syncthreads();   // the block and its first half's activations are in LDS, from every wave; block b - 1 is done with
            inputs(2 * c + 1, 1);
            if (b + 1 < blocks) rows.issue<false>(a0, to, wave);
            pf_products<T>(acc, lds.grid, stage, (const float*) (stage + DO), blk, 0, n, kq);
            wait_vm<0>();
            __syncthreads();
            if (b + 1 < blocks) {
                inputs(c + 1 == nc ? 0 : 2 * c + 2, 0);
                rows.issue<true>(a1, to + PF_WB, wave);
                next();
            }
            pf_products<T>(acc, lds.grid, stage + XB, (const float*) (stage + DO + 1024), blk, 1, n, kq);
            fold(blk);
        }
    }
}
template <int V> struct pf_int { static constexpr int value = V; };
// Straight-line products for the item's number of token tiles: only that many tiles' sums are live in the loop.
template <class F>
__device__ __forceinline__ void pf_tiles(u32 nt, F&& run) {
    switch ((nt + 15) / 16) {
        case 1: return run(pf_int<1>{});
        case 2: return run(pf_int<2>{});
        case 3: return run(pf_int<3>{});
        default: return run(pf_int<PF_TILES>{});
    }
}

// Work item blockIdx.y = (expert, first position) from prefill_group: gate and up rows [64 blockIdx.x, +64) of
// the expert against up to 64 of its pairs' tokens, SwiGLU (silu in f32, cpu_expert.rs:217), and H re-quantized per 32
// features: hq[pair][ff], hh the same codes times 2^-6 as f16, hd[pair][ff / 32].  eaddr[part * ne + e] / sh_addr[part] as in the planner's kernels.
// grid = (ff / 64, the bound on the number of items), block 512.
extern "C" __global__ void __launch_bounds__(512, 4) prefill_gate_up_iq3_s(const u64* eaddr, const u64* sh_addr, const u32* offs, const u32* list,
                                                                        const u32* items, const u16* xh, const float* xd, i8* hq, u16* hh, float* hd, u32 ne,
                                                                        u32 k, u32 npairs, u32 hidden, u32 ff) {
    constexpr u32 HP = 68;
    __shared__ __attribute__((aligned(16))) PfLds lds;   // the stages are afterwards the item's 64 x 64 block of H
    u8* stage = lds.stage;
    u32 *s_rows = lds.rows, *s_pairs = lds.pairs;
    static_assert(sizeof(lds.stage) >= 2 * PF_TOK * HP * sizeof(float), "H and the up sums reuse the staging area");
    const u32 tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const u32 n = lane & 15, kq = lane >> 4, rbx = blockIdx.x;
    const u32 rb = hidden / 256 * 110;
    if (blockIdx.y >= items[0]) return;
    const u32 e = items[1 + 2 * blockIdx.y], t0 = items[2 + 2 * blockIdx.y];
    if (e == ne && !sh_addr) return;
    const u32 first = offs[e], nt = min((u32) PF_TOK, offs[e + 1] - first - t0);
    pf_tables(lds.grid, tid);
    const u64 wg = uniform_u64(e < ne ? eaddr[e] : sh_addr[0]) + (u64) rbx * 64 * rb, wu = uniform_u64(e < ne ? eaddr[(u64) ne + e] : sh_addr[1]) + (u64) rbx * 64 * rb;
    if (tid < PF_TOK) {   // a place past the item's end has row 0, whose products are dropped
        const u32 p = tid < nt ? list[first + t0 + tid] : 0;
        s_pairs[tid] = p;
        s_rows[tid] = p < npairs ? p / k : p - npairs;
    }
    __syncthreads();   // s_rows and the table are written
    float (*hs)[HP] = (float (*)[HP]) stage;
    float (*us)[HP] = (float (*)[HP]) (stage + PF_TOK * HP * sizeof(float));
    pf_tiles(nt, [&](auto tiles) {
        constexpr int T = decltype(tiles)::value;
        pf_stream<T>(lds, wg, wu, 0, rb, hidden / 256, hidden / 256, xh, xd, s_rows, hidden, wave, lane, [&](u32, f32x4 (&sums)[T]) {
            // the staging area becomes H [token][feature]: up's sums go to the waves that hold gate's
            __syncthreads();
            if (wave >= 4) {
#pragma unroll
                for (int a = 0; a < T; a++) *(f32x4*) &us[16 * a + n][16 * (wave - 4) + 4 * kq] = sums[a];
            }
            __syncthreads();
            // H = silu(gate) * up for (token 16 a + n, features 16 wave + 4 kq + r)
            if (wave < 4) {
#pragma unroll
                for (int a = 0; a < T; a++) {
                    const f32x4 u = *(const f32x4*) &us[16 * a + n][16 * wave + 4 * kq];
                    f32x4 h;
#pragma unroll
                    for (int r = 0; r < 4; r++) h[r] = (sums[a][r] / (1.0f + expf(-sums[a][r]))) * u[r];
                    *(f32x4*) &hs[16 * a + n][16 * wave + 4 * kq] = h;
                }
            }
            __syncthreads();
        });
    });
    // per-32 quantization over features: a thread 8 of them, the four threads of a 32-block side by side
    const u32 t = tid >> 3, f = 8 * (tid & 7);
    if (t < nt) {
        float v[8], amax = 0.0f;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            v[i] = hs[t][f + i];
            amax = fmaxf(amax, fabsf(v[i]));
        }
        amax = fmaxf(amax, lane_xor<1>(amax, lane));
        amax = fmaxf(amax, lane_xor<2>(amax, lane));
        const float dd = amax / 127.0f;
        const float id = dd > 0.0f ? 1.0f / dd : 0.0f;
        u32 q[2] = {0, 0};
#pragma unroll
        for (int i = 0; i < 8; i++) {
            v[i] = fminf(127.0f, fmaxf(-127.0f, roundf(v[i] * id)));
            q[i / 4] |= ((u32) (int) v[i] & 0xffu) << (8 * (i % 4));
            v[i] *= 0x1p-6f;
        }
        const u64 at = (u64) s_pairs[t] * ff + rbx * 64 + f;
        *(u32x2*) (hq + at) = u32x2{q[0], q[1]};
        *(u32x4*) (hh + at) = u32x4{f16_pair(v[0], v[1]), f16_pair(v[2], v[3]), f16_pair(v[4], v[5]), f16_pair(v[6], v[7])};
        if ((tid & 3) == 0) hd[at / 32] = dd;
    }
}

// Work item blockIdx.y: down rows of the expert against its pairs' H: eo[pair][hidden], unweighted (cpu_expert.rs:316-339).
// A workgroup takes hidden / 128 / gridDim.x lots of 128 rows one after the other: its set-up is paid once, and the loads of a
// lot's first blocks are in flight while the lot before it is multiplied.
// grid = (a divisor of hidden / 128, the bound on the number of items), block 512.
extern "C" __global__ void __launch_bounds__(512, 4) prefill_down_iq3_s(const u64* eaddr, const u64* sh_addr, const u32* offs, const u32* list,
                                                                     const u32* items, const u16* hh, const float* hd, float* eo, u32 ne, u32 hidden,
                                                                     u32 ff) {
    __shared__ __attribute__((aligned(16))) PfLds lds;
    u32* s_pairs = lds.pairs;
    const u32 tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const u32 n = lane & 15, kq = lane >> 4;
    const u32 rb = ff / 256 * 110, per = hidden / 128 / gridDim.x, lot0 = blockIdx.x * per;
    if (blockIdx.y >= items[0]) return;
    const u32 e = items[1 + 2 * blockIdx.y], t0 = items[2 + 2 * blockIdx.y];
    if (e == ne && !sh_addr) return;
    const u32 first = offs[e], nt = min((u32) PF_TOK, offs[e + 1] - first - t0);
    pf_tables(lds.grid, tid);
    const u64 wd = uniform_u64(e < ne ? eaddr[2ull * ne + e] : sh_addr[2]) + (u64) lot0 * 128 * rb;
    if (tid < PF_TOK) s_pairs[tid] = tid < nt ? list[first + t0 + tid] : 0;
    __syncthreads();   // s_pairs and the table are written
    pf_tiles(nt, [&](auto tiles) {
        constexpr int T = decltype(tiles)::value;
        pf_stream<T>(lds, wd, wd + 64ull * rb, 128ull * rb, rb, ff / 256, per * (ff / 256), hh, hd, s_pairs, ff, wave, lane, [&](u32 lot, f32x4 (&sums)[T]) {
            const u32 row = (lot0 + lot) * 128 + wave * 16 + 4 * kq;
#pragma unroll
            for (int a = 0; a < T; a++)
                if (16 * a + n < nt) *(f32x4*) (eo + (u64) s_pairs[16 * a + n] * hidden + row) = sums[a];
        });
    });
}

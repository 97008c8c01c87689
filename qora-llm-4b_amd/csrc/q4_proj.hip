// q4_proj.hip -- Q4 projections (the GEMVs around the token mixer) for gfx950.
//
// A Q4Weight (gemv.rs:29-34) maps k inputs to n outputs.  Each input row is
// cut into groups of 32 output columns with one f16 scale (absmax / 7) and 16
// bytes of 4-bit codes q, value = scale * (q - 8); byte j of a group holds
// column 2j in its low nibble and 2j + 1 in its high nibble (quantize_q4,
// convert.rs:437-467).  The reference stores it row-major:
//   packed u8 [k][n/2], scales f16 [k][n/32].
// On the device a weight is kept tile-major (qm_q4_repack, once at load
// time, as the reference's wgpu loader repacks for its backend,
// gpu_loader.rs:82-106): column tiles of T = 16 columns (T = 8 when
// n < 4096, so that even a 2560-wide weight spreads over 320 workgroups),
//   codes u8 [n/T][k][T/2], gscales f16 [n/32][k],
// so that everything one output tile needs is one contiguous stream.
//
// qm_q4_gemv computes y = x W (gemv_q4, gemv.rs:451-467, inner loop
// :412-445) for one input row, for up to four weights that share x in one
// launch (a launch costs a few microseconds of fixed time, about what a
// 2560x4096 weight takes to stream).  Optional fusions, each what the
// reference does right around that gemv call:
//   - x <- rms_norm(x, gamma) first (1 + gamma, eps 1e-6; gemv.rs:571-579),
//     as before in_proj_* / q,k,v_proj and before the MLP (gemv.rs:740,893);
//   - y <- residual + x W (the residual adds after out_proj / o_proj and
//     down_proj, gemv.rs:889-890,896);
//   - qm_q4_gate_up: silu(x Wg) * (x Wu) for one tile of both weights per
//     workgroup (fused_gate_up_q4, gemv.rs:469-526);
//   - on the first weight, the DeltaNet conv1d step + SiLU (gemv.rs:744-772)
//     of the in_proj_qkv output, with its conv buffer shifted in place.
// One workgroup owns one column tile and all k rows, so the result needs
// no second pass: lane t takes rows t, t + 512, ..., and loads its 8 rows'
// codes, scales, x (and norm weights) before any arithmetic, at clamped
// rows so that no load waits behind a branch.  The T partial sums of every
// lane are reduced across the wave in registers (a transpose-reduce over
// lane swaps), then across the waves through LDS behind one barrier, in a
// fixed order (bit-reproducible run to run).  A weight costs ~1.7 VALU
// instructions: the codes enter the fma as f16 (see q4_halves) and as q
// itself, the -8 offset being applied once per lane through sum(scale * x).
// (With a v_cvt_f32_ubyteN per code, 2.4 instructions, the four launches of
// a layer took 0.4 us more: 2560 x 12288 6.45 -> 6.31 us, 9216 x 2560 7.15
// -> 7.02, 4096 x 2560 4.35 -> 4.26, the gate / up pair unchanged at 9.7,
// of which 1.9 are an empty launch and 4.3 the weights at 6.2 TB/s.)  A wave
// whose sums say that its operands left the codes' range (q4_in_range, 0.02
// us a launch) forms them again with the codes converted.
// The RMSNorm is applied by linearity: y = inv_rms * (x (1 + gamma)) W, so
// its sum of squares comes from the same x loads and the factor scales the
// column sums.
#include "qm_device.h"
#include "qm_q4_tiles.h"
#include <type_traits>
#include "qm_kernel_args.h"

#define Q4_THREADS 512
#define Q4_STEPS 8          // rows per lane in flight

template <int T> struct Q4Codes;                          // T/2 bytes of codes
template <> struct Q4Codes<16> { typedef uint2 type; };
template <> struct Q4Codes<8> { typedef uint32_t type; };
template <int T> struct Q4Pair;                           // two consecutive rows' codes
template <> struct Q4Pair<16> {
    typedef uint4 type;
    static QM_DEV uint2 half(uint4 v, int h) { return h ? make_uint2(v.z, v.w) : make_uint2(v.x, v.y); }
};
template <> struct Q4Pair<8> {
    typedef uint2 type;
    static QM_DEV uint32_t half(uint2 v, int h) { return h ? v.y : v.x; }
};

QM_DEV void q4_word(float* acc, uint32_t w, float se, float so) {  // 8 codes: columns 0..7 of acc
    q4_half2 h[4];
    q4_halves(w, h);
#pragma unroll
    for (int b = 0; b < 8; ++b) acc[b] = fmaf((float)h[b & 3][b >> 2], b & 1 ? so : se, acc[b]);
}
// acc += q * sx / QM_Q4_SUM
QM_DEV void q4_accumulate(float (&acc)[16], uint2 c, float sx) {
    const float se = sx * QM_Q4_EVEN, so = sx * QM_Q4_ODD;
    q4_word(acc, c.x, se, so);
    q4_word(acc + 8, c.y, se, so);
}
QM_DEV void q4_accumulate(float (&acc)[8], uint32_t c, float sx) { q4_word(acc, c, sx * QM_Q4_EVEN, sx * QM_Q4_ODD); }

// Whether the wave's column sums are those of operands within the f16 codes'
// range: one past it leaves every even column infinite or NaN, and the bits
// lost to subnormals matter only where every sum is tiny (beside larger ones
// they could break a rounding tie, no more).  Zeros are rows past k.
QM_DEV bool q4_in_range(float y, float u) {
    constexpr uint32_t LO = 0x17800000u, INF = 0x7f800000u;   // 2^-80
    const uint32_t a = __float_as_uint(y) & 0x7fffffffu, b = __float_as_uint(u) & 0x7fffffffu, m = a > b ? a : b;
    if (__builtin_expect(!__any(m - LO >= INF - LO), 1)) return true;
    return !__any(m >= INF) && (__any(m >= LO) || !__any(m));
}
// A lane's column partials with the codes converted to f32, for operands at
// the ends of f32's range: the rows and their order are those of q4_tile.
template <int T, int GROUP, int THREADS>
QM_DEV void q4_wide_partials(float (&acc)[T], const void* codes, const uint16_t* gsc, const float* x, const uint16_t* nw,
                             int K) {
    const uint32_t* words = reinterpret_cast<const uint32_t*>(codes);
#pragma unroll
    for (int j = 0; j < T; ++j) acc[j] = 0.0f;
#pragma unroll 1
    for (int i = 0;; ++i) {
        const int k = GROUP * (i / GROUP * THREADS + (int)threadIdx.x) + i % GROUP;
        if (k >= K) break;
        const float xn = nw ? x[k] * (1.0f + f16_to_f32(nw[k])) : x[k];
        const float sx = f16_to_f32(gsc[k]) * xn;
#pragma unroll
        for (int j = 0; j < T; ++j)
            acc[j] = fmaf((float)((words[(size_t)k * (T / 8) + j / 8] >> (4 * (j % 8))) & 15u), sx, acc[j]);
    }
}

// Wave-level sum of each of a lane's T column partials by transpose-reduce:
// each step pairs lane l with l ^ 32, ^16, ^8 (and ^4 for T = 16), and each
// lane keeps the half of its columns its side of the pair owns, summed with
// the partner's copy of them; then the remaining lane bits are summed.  At
// the end lane l holds the wave's total of column q4_col<T>(l) (the same in
// the 64 / T lanes that share it).  No LDS, no barrier; a fixed order, so
// the result is reproducible run to run.
QM_DEV float xor_swz4(float x) {            // the value of lane l ^ 4 (ds_swizzle bit mode)
    return __builtin_bit_cast(float, __builtin_amdgcn_ds_swizzle(__builtin_bit_cast(int, x), 0x101F));
}
// (n is a template parameter: as a runtime argument the compiler did not
// unroll these loops and indexed v through 16-way compare/select chains)
template <int N>
QM_DEV void halve32(float* v) {             // N values -> N/2: lanes < 32 keep 0..N/2-1
#pragma unroll
    for (int j = 0; j < N / 2; ++j) {
        const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[j]), __float_as_uint(v[j + N / 2]), false, false);
        v[j] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
}
template <int N>
QM_DEV void halve16(float* v) {             // even 16-lane rows keep 0..N/2-1
#pragma unroll
    for (int j = 0; j < N / 2; ++j) {
        const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v[j]), __float_as_uint(v[j + N / 2]), false, false);
        v[j] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
}
template <int BIT, int N>
QM_DEV void halve_dpp(float* v, int lane) {  // lanes with bit BIT clear keep 0..N/2-1
    const bool hi = (lane >> BIT) & 1;
#pragma unroll
    for (int j = 0; j < N / 2; ++j) {
        const float keep = hi ? v[j + N / 2] : v[j];
        const float send = hi ? v[j] : v[j + N / 2];
        const float got = BIT == 3 ? dpp_f32<0x128>(send) : xor_swz4(send);   // row_ror:8 = lane ^ 8
        v[j] = keep + got;
    }
}
template <int T> QM_DEV int q4_col(int lane) {
    return T == 16 ? 8 * ((lane >> 5) & 1) + 4 * ((lane >> 4) & 1) + 2 * ((lane >> 3) & 1) + ((lane >> 2) & 1)
                   : 4 * ((lane >> 5) & 1) + 2 * ((lane >> 4) & 1) + ((lane >> 3) & 1);
}
template <int T>
QM_DEV float q4_wave_reduce(float (&v)[T], int lane) {
    halve32<T>(v);
    halve16<T / 2>(v);
    halve_dpp<3, T / 4>(v, lane);
    float x;
    if (T == 16) {
        halve_dpp<2, 2>(v, lane);
        x = v[0];
    } else {
        x = v[0];
        x += xor_swz4(x);
    }
    x += dpp_f32<0x4E>(x);                  // lane ^ 2
    x += dpp_f32<0xB1>(x);                  // lane ^ 1
    return x;
}

// base[idx] with a 32-bit byte offset from a wave-uniform base, so the load
// takes the scalar-base + 32-bit vector-offset form (no 64-bit address
// arithmetic per lane)
template <class V>
QM_DEV V ld_off(const V* base, uint32_t idx) {
    return *reinterpret_cast<const V*>(reinterpret_cast<const char*>(base) + (size_t)(idx * (uint32_t)sizeof(V)));
}

template <bool GATE_UP, bool PAIR, bool NORM, int T, int STEPS, int THREADS>
QM_DEV void q4_tile(const Q4GemvArgs& A, int p, int tile, float (*red)[33]) {
    typedef typename Q4Codes<T>::type CodeT;
    const int tid = threadIdx.x;
    const int K = A.k;
    const int g = tile / (32 / T);                        // the tile's 32-column scale group
    const CodeT* codes = reinterpret_cast<const CodeT*>(A.codes[p]) + (size_t)tile * K;
    const uint16_t* gsc = A.gscales[p] + (size_t)g * K;
    const CodeT* codes_u = GATE_UP ? reinterpret_cast<const CodeT*>(A.codes[1]) + (size_t)tile * K : nullptr;
    const uint16_t* gsc_u = GATE_UP ? A.gscales[1] + (size_t)g * K : nullptr;
    // NORM (A.norm_w set, uniform over the launch) is a template parameter: a
    // load under a condition would wait for its data before the next step's
    // loads issue
    const uint16_t* nwp = A.norm_w;

    float acc[T], acc_u[GATE_UP ? T : 1];
#pragma unroll
    for (int j = 0; j < T; ++j) acc[j] = 0.0f;
#pragma unroll
    for (int j = 0; j < (GATE_UP ? T : 1); ++j) acc_u[j] = 0.0f;
    float bsum = 0.0f, bsum_u = 0.0f, ss = 0.0f;
    if (PAIR) {
        // two consecutive rows per load: their codes (2 x T/2 bytes), scales,
        // x values and norm weights are adjacent, so one load instruction of
        // twice the width takes both (k is even on this path)
        typedef typename Q4Pair<T>::type PairT;
        const int KP = K >> 1;
        const PairT* codes2 = reinterpret_cast<const PairT*>(codes);
        const PairT* codes2_u = reinterpret_cast<const PairT*>(codes_u);
        const uint32_t* gsc2 = reinterpret_cast<const uint32_t*>(gsc);
        const uint32_t* gsc2_u = reinterpret_cast<const uint32_t*>(gsc_u);
        const uint32_t* nwp2 = reinterpret_cast<const uint32_t*>(nwp);
        const float2* x2 = reinterpret_cast<const float2*>(A.x);
        constexpr int PS = STEPS / 2;
        for (int k0 = 0; k0 < KP; k0 += THREADS * PS) {
            PairT pk[PS], pu[GATE_UP ? PS : 1];
            uint32_t sc[PS], su[GATE_UP ? PS : 1], nw[PS];
            float2 xv[PS];
#pragma unroll
            for (int s = 0; s < PS; ++s) {
                const uint32_t kp = min((uint32_t)(k0 + tid + THREADS * s), (uint32_t)(KP - 1));
                pk[s] = ld_off(codes2, kp);
                sc[s] = ld_off(gsc2, kp);
                if (GATE_UP) {
                    pu[s] = ld_off(codes2_u, kp);
                    su[s] = ld_off(gsc2_u, kp);
                }
                xv[s] = ld_off(x2, kp);
                if (NORM) nw[s] = ld_off(nwp2, kp);
            }
            const bool full = k0 + THREADS * PS <= KP;
#pragma unroll
            for (int s = 0; s < PS; ++s) {
                if (!full && k0 + THREADS * s + (tid & ~63) >= KP) break;
                const bool ok = full || k0 + tid + THREADS * s < KP;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const float xl = ok ? (h ? xv[s].y : xv[s].x) : 0.0f;
                    ss = fmaf(xl, xl, ss);
                    const float xn = NORM ? xl * (1.0f + f16_to_f32((uint16_t)(nw[s] >> (16 * h)))) : xl;
                    const float sx = f16_to_f32((uint16_t)(sc[s] >> (16 * h))) * xn;
                    bsum += sx;
                    q4_accumulate(acc, Q4Pair<T>::half(pk[s], h), sx);
                    if (GATE_UP) {
                        const float sxu = f16_to_f32((uint16_t)(su[s] >> (16 * h))) * xn;
                        bsum_u += sxu;
                        q4_accumulate(reinterpret_cast<float(&)[T]>(acc_u), Q4Pair<T>::half(pu[s], h), sxu);
                    }
                }
            }
        }
    } else {
        for (int k0 = 0; k0 < K; k0 += THREADS * STEPS) {
            CodeT pk[STEPS], pu[GATE_UP ? STEPS : 1];
            uint16_t sc[STEPS], su[GATE_UP ? STEPS : 1], nw[STEPS];
            float xv[STEPS];
    #pragma unroll
            for (int s = 0; s < STEPS; ++s) {
                const uint32_t k = min((uint32_t)(k0 + tid + THREADS * s), (uint32_t)(K - 1));
                pk[s] = ld_off(codes, k);
                sc[s] = ld_off(gsc, k);
                if (GATE_UP) {
                    pu[s] = ld_off(codes_u, k);
                    su[s] = ld_off(gsc_u, k);
                }
                xv[s] = ld_off(A.x, k);
                if (NORM) nw[s] = ld_off(nwp, k);
            }
            const bool full = k0 + THREADS * STEPS <= K;    // workgroup-uniform: every row valid
    #pragma unroll
            for (int s = 0; s < STEPS; ++s) {
                // rows past k (wave-uniform except in the last wave) add nothing
                if (!full && k0 + THREADS * s + (tid & ~63) >= K) break;
                const float xl = full || k0 + tid + THREADS * s < K ? xv[s] : 0.0f;
                ss = fmaf(xl, xl, ss);
                const float xn = NORM ? xl * (1.0f + f16_to_f32(nw[s])) : xl;   // gemv.rs:575 but inv_rms
                const float sx = f16_to_f32(sc[s]) * xn;                           // gemv.rs:429: scale * x_k
                bsum += sx;
                q4_accumulate(acc, pk[s], sx);
                if (GATE_UP) {
                    const float sxu = f16_to_f32(su[s]) * xn;
                    bsum_u += sxu;
                    q4_accumulate(reinterpret_cast<float(&)[T]>(acc_u), pu[s], sxu);
                }
            }
        }
    }

    // Column sums: each wave reduces its lanes' partials in registers (the
    // -8 code offset applied through the scale * x sums), writes one value
    // per column, and after one barrier thread j < T adds the THREADS / 64
    // waves' values in order.  x's sum of squares for the RMSNorm rides along.
    const int lane = tid & 63, wv = tid >> 6;
#pragma unroll
    for (int j = 0; j < T; ++j) acc[j] = fmaf(QM_Q4_SUM, acc[j], -8.0f * bsum);
    float cs = q4_wave_reduce<T>(acc, lane);
    float cs_u = 0.0f;
    if (GATE_UP) {
#pragma unroll
        for (int j = 0; j < T; ++j) acc_u[j] = fmaf(QM_Q4_SUM, acc_u[j], -8.0f * bsum_u);
        cs_u = q4_wave_reduce<T>(reinterpret_cast<float(&)[T]>(acc_u), lane);
    }
    const float ssw = NORM ? wave_sum64(ss) : 0.0f;
    auto publish = [&] {
        if ((lane & (64 / T - 1)) == 0) {
            red[wv][q4_col<T>(lane)] = cs;
            if (GATE_UP) red[wv][16 + q4_col<T>(lane)] = cs_u;
        }
    };
    publish();
    if (lane == 0) red[wv][32] = ssw;
    if (!q4_in_range(cs, cs_u)) {
        auto wide = [&](const CodeT* c, const uint16_t* sc, float b) {
            float w[T];
            q4_wide_partials<T, PAIR ? 2 : 1, THREADS>(w, c, sc, A.x, NORM ? nwp : nullptr, K);
#pragma unroll
            for (int j = 0; j < T; ++j) w[j] = fmaf(-8.0f, b, w[j]);
            return q4_wave_reduce<T>(w, lane);
        };
        cs = wide(codes, gsc, bsum);
        if (GATE_UP) cs_u = wide(codes_u, gsc_u, bsum_u);
        publish();
    }
    __syncthreads();
    float y = 0.0f, u = 0.0f, sst = 0.0f;
    if (tid < T) {
#pragma unroll
        for (int w = 0; w < THREADS / 64; ++w) {
            y += red[w][tid];
            if (GATE_UP) u += red[w][16 + tid];
            sst += red[w][32];
        }
    }
    // gemv.rs:573: 1 / sqrt(mean(x^2) + 1e-6)
    const float inv = NORM ? 1.0f / sqrtf(sst / (float)K + 1e-6f) : 1.0f;
    y *= inv;
    if (GATE_UP) {
        u *= inv;
        // gemv.rs:524: (g / (1 + exp(-g))) * u
        if (tid < T) A.y[0][T * (size_t)tile + tid] = (y / (1.0f + expf(-y))) * u;
    } else if (tid < T) {
        const size_t c = T * (size_t)tile + tid;
        float v = A.residual[p] ? A.residual[p][c] + y : y;
        if (p == 0 && A.conv_buf) {
            // gemv.rs:744-772 on the in_proj_qkv output: causal depthwise
            // conv over the buffer (oldest .. newest) and v, buffer shift,
            // SiLU
            float* buf = A.conv_buf + c * 3;
            const float4 w = *reinterpret_cast<const float4*>(A.conv_w + c * 4);
            const float b0 = buf[0], b1 = buf[1], b2 = buf[2];
            const float s = conv_taps4(b0, b1, b2, v, w);
            buf[0] = b1;
            buf[1] = b2;
            buf[2] = v;
            v = silu_f(s);
        }
        A.y[p][c] = v;
    }
}

template <bool GATE_UP, bool NORM, int STEPS, int THREADS>
QM_DEV void q4_tile_pick(const Q4GemvArgs& A, int p, int tile, float (*red)[33]) {
    if (A.k & 1) {
        if (A.tile[p] == 16) q4_tile<GATE_UP, false, NORM, 16, STEPS, THREADS>(A, p, tile, red);
        else q4_tile<GATE_UP, false, NORM, 8, STEPS, THREADS>(A, p, tile, red);
    } else {
        if (A.tile[p] == 16) q4_tile<GATE_UP, true, NORM, 16, STEPS, THREADS>(A, p, tile, red);
        else q4_tile<GATE_UP, true, NORM, 8, STEPS, THREADS>(A, p, tile, red);
    }
}

template <bool GATE_UP, int STEPS, int THREADS, bool WITH_NORM = true>
QM_DEV void q4_gemv_body(const Q4GemvArgs& A) {
    __shared__ float red[THREADS / 64][33];   // per wave: column sums (gate, up), x's sum of squares
    // which weight: workgroups wstart[p] .. wstart[p+1]-1 are weight p's
    // tiles (gate / up: weights 0 and 1 share the tile index)
    int p = 0;
    if (!GATE_UP) {
#pragma unroll
        for (int q = 1; q < QM_Q4_MAX_OUT; ++q)
            if (q < A.count && (int)blockIdx.x >= A.wstart[q]) p = q;
    }
    const int tile = (int)blockIdx.x - A.wstart[p];
    if (WITH_NORM && A.norm_w) q4_tile_pick<GATE_UP, WITH_NORM, STEPS, THREADS>(A, p, tile, red);
    else q4_tile_pick<GATE_UP, false, STEPS, THREADS>(A, p, tile, red);
}

extern "C" __global__ __launch_bounds__(Q4_THREADS) void qm_q4_gemv(Q4GemvArgs A) {
    q4_gemv_body<false, Q4_STEPS, Q4_THREADS>(A);
}

// 256 threads, 10 rows (5 row pairs) per lane: one load round at k = 2560,
// and at 140 VGPRs three workgroups per CU, so the 576 tiles of the 2560 x
// 9216 gate / up pair are resident in one dispatch round (the 512-thread form
// fitted two per CU and ran 3% slower per model token).
extern "C" __global__ __launch_bounds__(256) void qm_q4_gate_up(Q4GemvArgs A) {
    q4_gemv_body<true, 10, 256>(A);
}

// Shape-fitted forms.  A launch's workgroups should all be resident at once
// (a second dispatch round repeats the whole load -> reduce latency), and a
// lane's rows should come in as few load rounds as possible:
//   k <= 2560 (the hidden size): 256 threads of 10 rows, one load round, 87
//     VGPRs (five workgroups per CU, 1280 slots for the 776 tiles of the
//     fused DeltaNet input projections);
//   k <= 9216 without a norm (the MLP's down_proj): 18 rows per lane, one
//     load round, 116 VGPRs (two workgroups per CU, 512 slots for 320
//     tiles); the host sends a launch with a norm to the general form.
// (512-thread forms of 5 rows for k <= 2560, of 18 or 12 rows at 256 threads
// for down_proj, and of 16 at 256 threads for the general case all measured
// slower over a model token.)
extern "C" __global__ __launch_bounds__(256)
void qm_q4_gemv_hidden(Q4GemvArgs A) {
    q4_gemv_body<false, 10, 256>(A);
}
extern "C" __global__ __launch_bounds__(Q4_THREADS) __attribute__((amdgpu_waves_per_eu(4)))
void qm_q4_gemv_inter(Q4GemvArgs A) {
    q4_gemv_body<false, 18, Q4_THREADS, false>(A);
}

// Reference layout -> tile-major.  Workgroup = 64 rows x 16 groups: each
// thread reads one 16-byte group block and one scale (consecutive along a
// row), and writes the block's 32 / T tile slices (consecutive along k
// within a tile: 64 rows x T/2 bytes).
extern "C" __global__ __launch_bounds__(256) void qm_q4_repack(Q4RepackArgs A) {
    __shared__ uint4 tc[16][65];
    __shared__ uint16_t ts[16][66];
    const int tid = threadIdx.x;
    const int G = A.n / 32, T = A.tile;
    const int gb = blockIdx.x % ((G + 15) / 16), kb = blockIdx.x / ((G + 15) / 16);
    const int k0 = kb * 64, g0 = gb * 16;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        const int r = p * 16 + (tid >> 4), j = tid & 15;
        const int k = k0 + r, g = g0 + j;
        if (k < A.k && g < G) {
            tc[j][r] = *reinterpret_cast<const uint4*>(A.packed + (size_t)k * (A.n / 2) + 16 * (size_t)g);
            ts[j][r] = A.scales[(size_t)k * G + g];
        }
    }
    __syncthreads();
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        const int j = p * 4 + (tid >> 6), r = tid & 63;
        const int k = k0 + r, g = g0 + j;
        if (k < A.k && g < G) {
            const uint4 v = tc[j][r];
            if (T == 16) {
                uint2* dst = reinterpret_cast<uint2*>(A.codes);
                dst[(size_t)(2 * g) * A.k + k] = make_uint2(v.x, v.y);
                dst[(size_t)(2 * g + 1) * A.k + k] = make_uint2(v.z, v.w);
            } else {
                uint32_t* dst = reinterpret_cast<uint32_t*>(A.codes);
                dst[(size_t)(4 * g) * A.k + k] = v.x;
                dst[(size_t)(4 * g + 1) * A.k + k] = v.y;
                dst[(size_t)(4 * g + 2) * A.k + k] = v.z;
                dst[(size_t)(4 * g + 3) * A.k + k] = v.w;
            }
            A.gscales[(size_t)g * A.k + k] = ts[j][r];
        }
    }
}

// ---------------------------------------------------------------------------
// Prefill: C[m][n] = X[m][k] W on MFMA (gemm_q4, gemv.rs:529-542, for
// seq_len > 1).  X is f16 (qm_rms_norm_f16 produces it from the f32 hidden
// state, fusing the layer's RMSNorm) or bf16 (the mixer outputs and the
// MLP's silu(g) * u).  W stays Q4 in HBM and in LDS and is dequantized into
// the MFMA operand registers: s * (q - 8) rounded once to f16 and, for a bf16
// X, on to bf16.  An f16 X runs v_mfma_f32_16x16x32_f16; a bf16 X is used as
// it is and runs v_mfma_f32_16x16x32_bf16, so it keeps fp32's range.
//
// Operand form.  A wave computes 16 MI rows x 16 NJ columns, and lane
// fr = lane & 15 of its fragment j holds column NJ fr + j.  The codes a lane
// needs of one row of k are then NJ neighbouring nibbles of one code word,
// and its outputs are NJ neighbouring columns, stored straight from the
// accumulators (16 bytes of fp32 at NJ = 4).
//
// Staging.  64 rows of k are a stage: x rows, raw codes and scales are copied
// to LDS by DMA, no registers and no LDS store instructions, each instruction
// covering whole 128-byte lines (an x operand read straight from global
// memory has 16 rows in 16 neighbouring lanes, which the memory path takes
// one lane at a time: measured 60 cache accesses per load instruction, the L1
// at one access per cycle the whole launch).  16-byte chunks are xor-swizzled
// in each row or tile so that the operand reads meet no bank conflict
// (SQ_LDS_BANK_CONFLICT 0).  One barrier per stage where the waves of a
// k-group share its x rows (WN > 1), none where a k-group is one wave.
//
// What bounds it.  Large m: issue slots.  Per step of 32 rows a 128 x 64 wave
// tile issues 32 MFMAs and ~80 VALU instructions (1.75 per weight pair and
// addressing), and a probe shows two VALU instructions per 16-cycle MFMA are
// free and each further one costs four cycles; timing copies put the
// dequantization at 28 us and the DMA at 28 us of 160 us (4096 x 2560 x
// 8192), without both and the barrier 109 us, which is what the MFMAs alone
// take.  Few rows: the chain of stages, ~0.45 us each for the smallest tile;
// so k is split over the waves of a workgroup (WK groups, their partial tiles
// added in group order through LDS at the end) until there is a workgroup
// for every CU.
//
// Measured against the form it replaces (codes dequantized once per
// workgroup into LDS, 128 x 256 tiles, one barrier per 32 rows), us, same
// box, rotating weights:
//   m x k x n            before    now
//   48 x 2560 x 8192       39.4    6.9     (DeltaNet in_proj_qkv)
//   48 x 9216 x 2560      141.9   13.3     (down_proj, bf16 x)
//   300 x 9216 x 2560     140     33
//   700 x 4096 x 2560      64     28       (o_proj, bf16 x)
//   4096 x 2560 x 8192    187    151       (1.14 PFLOP/s)
//   4096 x 9216 x 2560    271    235
//   4096 x 2560 x 32        9.9    5.1     (in_proj_a / b)
//   4096 x 2560 x 9216 gate/up  406    331  (1.17 PFLOP/s)
// Tried and no faster: dequantizing the next step's operand between the
// MFMAs of this one (explicit interleave; 0-3% either way), two LDS stages
// instead of three (0-2%), and reading x and codes without LDS (3-4 x slower
// from 300 rows on, for the access count above).
// ---------------------------------------------------------------------------
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

// An f16 pair as a bf16 pair, each rounded to nearest even (the f16 values
// are exact in fp32, so this is one rounding of each).
__device__ __forceinline__ uint32_t f16x2_to_bf16x2(half2 h) {
    const bf16x2 b = bf16x2{(__bf16)(float)h[0], (__bf16)(float)h[1]};
    return __builtin_bit_cast(uint32_t, b);
}

// LDS of one k-group and stage: x rows [16 MI][64] (chunk c of row r at slot
// c ^ (r & 7)), then per wave the codes of its 16 NJ columns x 64 rows and
// its scales [NJ / 2][64] (256 bytes).
template <int MI, int NJ, int WN, int WK, int NST>
struct Q4GemmLds {
    static constexpr int X = 16 * MI * 128, C = 512 * NJ, S = 256;
    static constexpr int STAGE = X + WN * (C + S);
    static constexpr int BYTES = WK * NST * STAGE;
};

// BIG: 64-bit lane offsets (k above QM_Q4_GEMM_MAX_K32).
template <bool XBF16, bool GU, int MI, int NJ, int WN, int WK, int NST, int T, bool BIG>
__device__ __forceinline__ void q4_gemm_loop(const Q4GemmArgs& A, int m0, int n0, char* smem, floatx4 (&acc)[MI][NJ]) {
    using L = Q4GemmLds<MI, NJ, WN, WK, NST>;
    using off_t = std::conditional_t<BIG, uint64_t, uint32_t>;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wn = w % WN, wk = w / WN;
    const int lane = threadIdx.x & 63, fr = lane & 15, kg = lane >> 4;
    const off_t K = A.k;
    constexpr int WO = GU && WN > 1 ? WN / 2 : WN;         // waves side by side over the output columns
    constexpr int KG = GU && WN == 1 ? WK / 2 : WK;        // k-groups per weight
    const bool up = GU && (WN > 1 ? wn >= WO : wk >= KG);
    const int nw = n0 + 16 * NJ * (wn % WO);               // the wave's first column
    constexpr int CPT = T == 16 ? 32 : 16;                 // 16-byte chunks of a tile per stage
    // this k-group's stages t0 .. t1 - 1 of nk 32-row steps in all
    const int nk = A.k / 32, ns = (nk + 1) / 2;
    const int g = wk % KG, t0 = (int)((int64_t)ns * g / KG), t1 = (int)((int64_t)ns * (g + 1) / KG);
    const int iters = (ns + KG - 1) / KG;

    // Lane offsets of the wave's DMA instructions, rows, tiles and groups
    // past the matrix clamped to its last; *back: what a lane of the second
    // 32 rows steps back where the stage has only the first.
    const int tlast = A.n / T - 1, tb = min(nw / T, tlast);
    const char* cbase = reinterpret_cast<const char*>(up ? A.codes2 : A.codes) + (size_t)tb * A.k * (T / 2);
    off_t co[NJ / 2];
    uint32_t cback[NJ / 2];
#pragma unroll
    for (int q = 0; q < NJ / 2; ++q) {
        const int tl = (64 * q + lane) / CPT, ch = ((64 * q + lane) % CPT) ^ (T == 16 ? tl & 3 : tl & 7);
        co[q] = (off_t)(min(nw / T + tl, tlast) - tb) * K * (T / 2) + ch * 16;
        cback[q] = ch >= CPT / 2 ? 32 * (T / 2) : 0;
    }
    const int glast = A.n / 32 - 1, gb = min(nw / 32, glast);
    const char* sbase = reinterpret_cast<const char*>(up ? A.gscales2 : A.gscales) + (size_t)gb * A.k * 2;
    const off_t so = ((off_t)(min(nw / 32 + (NJ == 4 ? lane / 32 : 0), glast) - gb) * K + 2 * (lane % 32)) * 2;
    const uint32_t sback = lane % 32 >= 16 ? 64 : 0;
    const char* xbase = reinterpret_cast<const char*>(A.x + (size_t)m0 * A.k);
    constexpr int NX = (2 * MI + WN - 1) / WN;             // x instructions (8 rows each) of this wave
    off_t xo[NX];
    const uint32_t xch = (lane & 7) ^ (lane >> 3), xback = xch >= 4 ? 64 : 0;
#pragma unroll
    for (int q = 0; q < NX; ++q) {
        const int r = 8 * min(wn * NX + q, 2 * MI - 1) + (lane >> 3);
        xo[q] = (off_t)min(r, A.m - 1 - m0) * K * 2 + xch * 16;
    }
    constexpr int PER = NX + NJ / 2 + 1;                   // DMA instructions per wave and stage
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem + wk * NST * L::STAGE;
    const char* sm = smem + wk * NST * L::STAGE;
    auto dma = [](const char* base, off_t off, uint32_t lds) {
        if constexpr (BIG) dma16(base + off, lds);
        else dma16_off(base, off, lds);
    };
    auto issue = [&](int t, int buf) {
        const bool half = 2 * t + 1 >= nk;                 // the last step of an odd count has no second one
        const uint32_t lx = lds0 + buf * L::STAGE, lc = lx + L::X + wn * (L::C + L::S);
#pragma unroll
        for (int q = 0; q < NX; ++q)
            dma(xbase + (size_t)t * 128, xo[q] - (half ? xback : 0), lx + 1024 * min(wn * NX + q, 2 * MI - 1));
#pragma unroll
        for (int q = 0; q < NJ / 2; ++q)
            dma(cbase + (size_t)t * (64 * (T / 2)), co[q] - (half ? cback[q] : 0), lc + 1024 * q);
        const off_t s = so - (half ? sback : 0);
        if constexpr (BIG) dma4(sbase + (size_t)t * 128 + s, lc + L::C);
        else dma4_off(sbase + (size_t)t * 128, s, lc + L::C);
    };

    const int mytile = (NJ * fr) / T;
    const uint32_t sel = 0x0c040c00u + 0x00010001u * (((NJ * fr) % 8) / 2);   // byte of the lane's first column pair
    // the f16 exponent pattern 0x6400 (1024) of each half, held in a VGPR so
    // that masking a nibble pair into it is one v_and_or_b32 (the mask is the
    // instruction's one literal)
    uint32_t vmagic;
    asm volatile("v_mov_b32 %0, 0x64006400" : "=v"(vmagic));

    // the MFMAs of rows 32 h .. +31 of a stage
    auto step = [&](const char* sx, const char* sc, int h) {
        uint32_t c[8];                                     // the lane's code word of rows 32 h + 8 kg .. +7
        if constexpr (T == 16) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint32_t* p = reinterpret_cast<const uint32_t*>(
                    sc + (mytile * CPT + 16 * h + 4 * kg + (r ^ (mytile & 3))) * 16) + ((NJ * fr) % 16) / 8;
                c[2 * r] = p[0];
                c[2 * r + 1] = p[2];
            }
        } else {
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                const uint4 v = *reinterpret_cast<const uint4*>(sc + (mytile * CPT + ((8 * h + 2 * kg + r) ^ (mytile & 7))) * 16);
                c[4 * r] = v.x; c[4 * r + 1] = v.y; c[4 * r + 2] = v.z; c[4 * r + 3] = v.w;
            }
        }
        const uint4 sv = *reinterpret_cast<const uint4*>(sc + L::C + (NJ * fr / 32) * 128 + 64 * h + 16 * kg);
        const uint32_t s4[4] = {sv.x, sv.y, sv.z, sv.w};
        // Columns 2 q, 2 q + 1 of the lane are the low and high nibbles of
        // one byte of each row.  v_perm_b32 puts that byte of a row pair in
        // the two halves; masked into 0x6400 they are 1024 + c and 1024 + 16
        // c, and 1024 + c - 1032 and (1024 + 16 c) / 16 - 72 are c - 8
        // exactly; times s is the one rounding (the same bits as rounding s *
        // (c - 8) from fp32).
        uint32_t b[NJ][4];
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const half2 s2 = __builtin_bit_cast(half2, s4[p]);
            auto put = [&](int j, half2 q8) {
                const half2 v = q8 * s2;
                b[j][p] = XBF16 ? f16x2_to_bf16x2(v) : __builtin_bit_cast(uint32_t, v);
            };
#pragma unroll
            for (int q = 0; q < NJ / 2; ++q) {
                const uint32_t wd = __builtin_amdgcn_perm(c[2 * p + 1], c[2 * p], sel + 0x00010001u * q);
                put(2 * q, __builtin_bit_cast(half2, (wd & 0x000f000fu) | vmagic) - half2{1032.0f16, 1032.0f16});
                put(2 * q + 1, __builtin_elementwise_fma(__builtin_bit_cast(half2, (wd & 0x00f000f0u) | vmagic),
                                                         half2{0.0625f16, 0.0625f16}, half2{-72.0f16, -72.0f16}));
            }
        }
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            const uint4 a = *reinterpret_cast<const uint4*>(sx + i * 2048 + fr * 128 + (((4 * h + kg) ^ (fr & 7)) << 4));
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const uint4 bj = make_uint4(b[j][0], b[j][1], b[j][2], b[j][3]);
                if constexpr (XBF16)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        __builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, bj), acc[i][j], 0, 0, 0);
                else
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                        __builtin_bit_cast(half8, a), __builtin_bit_cast(half8, bj), acc[i][j], 0, 0, 0);
            }
        }
    };
#pragma unroll
    for (int p = 0; p < NST - 1; ++p)
        if (t0 + p < t1) issue(t0 + p, p);
    int buf = 0;
    // Stage t has landed once at most the younger stage's DMAs are left; the
    // barrier makes that true of every wave's part, and says that every wave
    // has read stage t - 1 (lgkmcnt: its reads have returned), whose buffer
    // is filled next.  A k-group of one wave (WN = 1) fills and reads its own
    // buffers only: its waits are enough, and its waves drift apart, one's
    // dequantization beside another's MFMAs.
    static_assert(NST == 2 || NST == 3, "at most one younger stage in flight");
    auto next = [&](int t) {
        if (NST == 3 && t + 1 < t1) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"(PER) : "memory");
        else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        if (WN > 1) asm volatile("s_barrier" ::: "memory");
        if (t + NST - 1 < t1) issue(t + NST - 1, buf == 0 ? NST - 1 : buf - 1);
    };
    // No branch around the MFMAs inside the loop: the accumulators would be
    // copied at every merge.
    const bool odd = t1 > t0 && 2 * t1 > nk;               // the range ends in a single step
    const int tf = odd ? t1 - 1 : t1;
    for (int t = t0; t < tf; ++t) {
        next(t);
        const char* sx = sm + buf * L::STAGE;
        const char* sc = sx + L::X + wn * (L::C + L::S);
        step(sx, sc, 0);
        step(sx, sc, 1);
        buf = buf == NST - 1 ? 0 : buf + 1;
    }
    if (odd) {
        next(tf);
        const char* sx = sm + buf * L::STAGE;
        step(sx, sx + L::X + wn * (L::C + L::S), 0);
    }
    // k-groups with fewer stages keep step
    for (int it = t1 - t0; WN > 1 && it < iters; ++it) asm volatile("s_barrier" ::: "memory");
}

// GU: the gate/up form.  Waves 0 .. WN/2 - 1 of a k-group take the gate
// weight's columns and the others the same columns of the up weight (WN = 1:
// the first half of the k-groups the gate weight, the second half the up
// weight); the epilogue writes silu(g) * u as bf16 (whose range, unlike
// f16's, holds any product of the fp32 accumulators).
template <bool XBF16, bool GU, int MI, int NJ, int WN, int WK, int NST, bool BIG = false>
__device__ __forceinline__ void q4_gemm_body(const Q4GemmArgs& A) {
    using L = Q4GemmLds<MI, NJ, WN, WK, NST>;
    static_assert(!GU || (WN == 1 ? WK : WN) % 2 == 0, "gate/up: half of the waves take the up weight");
    static_assert(NJ == 2 || NJ == 4, "a lane's columns are one or two bytes of a row");
    constexpr int WO = GU && WN > 1 ? WN / 2 : WN, WAVES = WN * WK;
    constexpr int KG = GU && WN == 1 ? WK / 2 : WK;        // k-groups per weight
    constexpr bool DIRECT = WK == 1 && !GU;                // one wave holds the whole sum of its outputs
    constexpr int KB = WAVES * NJ;                         // KB of partials per 16 rows
    constexpr int RB = L::BYTES > 65536 ? 64 : 32;         // KB of partials per round
    constexpr int IR = KB * MI <= RB ? MI : (RB / KB > 1 ? RB / KB : 1);
    constexpr int SMEM = DIRECT || L::BYTES > KB * IR * 1024 ? L::BYTES : KB * IR * 1024;
    __shared__ __attribute__((aligned(1024))) char smem[SMEM];
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int wn = w % WN, wk = w / WN;
    constexpr int NC = 16 * NJ * WO;
    // consecutive workgroups walk n within one row block: its x rows are
    // reused from L2 across its column tiles
    const int nbn = (A.n + NC - 1) / NC;
    const int bm = (int)(blockIdx.x / (uint32_t)nbn), bn = (int)(blockIdx.x % (uint32_t)nbn);
    const int m0 = bm * 16 * MI, n0 = bn * NC;
    floatx4 acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    if (A.tile == 16) q4_gemm_loop<XBF16, GU, MI, NJ, WN, WK, NST, 16, BIG>(A, m0, n0, smem, acc);
    else q4_gemm_loop<XBF16, GU, MI, NJ, WN, WK, NST, 8, BIG>(A, m0, n0, smem, acc);

    // n % 32 == 0 and col % NJ == 0: a lane's NJ columns are all in or all out
    auto store = [&](int row, int col, float (&y)[NJ]) {
        const size_t o = (size_t)row * A.n + col;
        if (!GU && A.residual) {
#pragma unroll
            for (int j = 0; j < NJ; ++j) y[j] += A.residual[o + j];
        }
        if (GU || A.y_bf16) {
#pragma unroll
            for (int j = 0; j < NJ; j += 2)
                *reinterpret_cast<uint32_t*>(A.y_bf16 + o + j) = pack_bf16x2(y[j], y[j + 1]);
        } else {
#pragma unroll
            for (int j = 0; j < NJ; ++j) A.y[o + j] = y[j];
        }
    };
    if constexpr (DIRECT) {
        const int col = n0 + 16 * NJ * wn + NJ * (lane & 15);
        if (col >= A.n) return;
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int row = m0 + 16 * i + 4 * (lane >> 4) + e;
                float y[NJ];
#pragma unroll
                for (int j = 0; j < NJ; ++j) y[j] = acc[i][j][e];
                if (row < A.m) store(row, col, y);
            }
    } else {
        // the k-groups' partial tiles meet where the stages were, IR row
        // tiles a round, and are added in group order
        float (*part)[WK][WN][4][64][NJ] = reinterpret_cast<float (*)[WK][WN][4][64][NJ]>(smem);
#pragma unroll
        for (int i0 = 0; i0 < MI; i0 += IR) {
            __syncthreads();
#pragma unroll
            for (int i = 0; i < IR; ++i)
                if (i0 + i < MI)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
#pragma unroll
                        for (int j = 0; j < NJ; ++j) part[i][wk][wn][e][lane][j] = acc[i0 + i][j][e];
            __syncthreads();
            for (int it = tid; it < IR * WO * 256; it += WAVES * 64) {
                const int l = it & 63, e = (it >> 6) & 3, c = (it >> 8) % WO, i = (it >> 8) / WO;
                const int row = m0 + 16 * (i0 + i) + 4 * (l >> 4) + e, col = n0 + 16 * NJ * c + NJ * (l & 15);
                if (i0 + i >= MI || row >= A.m || col >= A.n) continue;
                auto sum = [&](int g0, int v, float (&y)[NJ]) {
#pragma unroll
                    for (int j = 0; j < NJ; ++j) y[j] = part[i][g0][v][e][l][j];
#pragma unroll
                    for (int g = 1; g < KG; ++g)
#pragma unroll
                        for (int j = 0; j < NJ; ++j) y[j] += part[i][g0 + g][v][e][l][j];
                };
                float y[NJ];
                sum(0, c, y);
                if constexpr (GU) {
                    float u[NJ];
                    if constexpr (WN == 1) sum(KG, c, u);
                    else sum(0, WO + c, u);
#pragma unroll
                    for (int j = 0; j < NJ; ++j) y[j] = silu_fast(y[j]) * u[j];
                }
                store(row, col, y);
            }
        }
    }
}

#define Q4_GEMM(NAME, XB, GU, MI, NJ, WN, WK, NST, OCC, ...)                                       \
    extern "C" __global__ __launch_bounds__(64 * WN * WK, OCC) void NAME(Q4GemmArgs A) {          \
        q4_gemm_body<XB, GU, MI, NJ, WN, WK, NST, ##__VA_ARGS__>(A);                               \
    }
#define Q4_GEMM_PLAIN(MI, NJ, WN, WK, NST, OCC, ...)                                               \
    Q4_GEMM(qm_q4_gemm_f16_m##MI##n##NJ##w##WN##k##WK, false, false, MI, NJ, WN, WK, NST, OCC)     \
    Q4_GEMM(qm_q4_gemm_bf16_m##MI##n##NJ##w##WN##k##WK, true, false, MI, NJ, WN, WK, NST, OCC)
#define Q4_GEMM_GATE_UP(MI, NJ, WN, WK, NST, OCC, ...)                                             \
    Q4_GEMM(qm_q4_gemm_gu_f16_m##MI##n##NJ##w##WN##k##WK, false, true, MI, NJ, WN, WK, NST, OCC)   \
    Q4_GEMM_GATE_UP_BF16(MI, NJ, WN, WK, NST, OCC)
#define Q4_GEMM_GATE_UP_BF16(MI, NJ, WN, WK, NST, OCC, ...)                                        \
    Q4_GEMM(qm_q4_gemm_gu_bf16_m##MI##n##NJ##w##WN##k##WK, true, true, MI, NJ, WN, WK, NST, OCC)
QM_Q4_TILES_ONE_WAVE(Q4_GEMM_PLAIN)
QM_Q4_TILES_GATE_UP_BF16(Q4_GEMM_PLAIN)
QM_Q4_TILES_PAIRED(Q4_GEMM_PLAIN)
QM_Q4_TILES_ODD(Q4_GEMM_PLAIN)
QM_Q4_TILES_ONE_WAVE(Q4_GEMM_GATE_UP)
QM_Q4_TILES_GATE_UP_BF16(Q4_GEMM_GATE_UP_BF16)
QM_Q4_TILES_PAIRED(Q4_GEMM_GATE_UP)
Q4_GEMM(qm_q4_gemm_f16_big, false, false, 1, 2, 1, 8, 3, 4, true)
Q4_GEMM(qm_q4_gemm_bf16_big, true, false, 1, 2, 1, 8, 3, 4, true)
Q4_GEMM(qm_q4_gemm_gu_f16_big, false, true, 1, 2, 1, 8, 3, 4, true)
Q4_GEMM(qm_q4_gemm_gu_bf16_big, true, true, 1, 2, 1, 8, 3, 4, true)

// rms_norm (1 + gamma, eps 1e-6; gemv.rs:571-579) of each of m rows of f32
// x [m][k], written as the f16 input of qm_q4_gemm; without a norm weight,
// the plain f16 conversion.  One workgroup per row.  Rows of up to NV x 1024
// values stay in registers between the sum of squares and the output, with
// the norm weights requested beside them: one memory round trip, where
// reading the row again cost a second.  Longer rows are read twice.  NV is 1,
// 2 or 4 by the row's length, and lanes past its end load nothing: with four
// loads in every lane a row of up to 1024 values took up to 1.7 times as long
// as read twice.  Replayed graph, us, read twice / four loads / now:
//   8192 x 64     5.6 / 9.4 / 5.4      4096 x 1280   6.2 / 7.5 / 5.8
//   8192 x 1024  10.7 / 11.8 / 10.0    300 x 2560    2.9 / 2.6 / 2.5
//   4096 x 2560  12.9 / 10.7 / 10.8    8192 x 4096  42.0 / 29.1 / 29.3
template <int NV>
__device__ __forceinline__ void rms_norm_f16_body(const RmsNormArgs& A) {
    __shared__ float red[4];
    const int tid = threadIdx.x, row = blockIdx.x;
    const float* x = A.x + (size_t)row * A.k;
    uint16_t* out = A.out + (size_t)row * A.k;
    float ss = 0.0f;
    auto square = [&](float4 v) {
        ss = fmaf(v.x, v.x, ss); ss = fmaf(v.y, v.y, ss); ss = fmaf(v.z, v.z, ss); ss = fmaf(v.w, v.w, ss);
    };
    auto total = [&]() {
        ss = wave_sum64(ss);
        if ((tid & 63) == 0) red[tid >> 6] = ss;
        __syncthreads();
        return A.norm_w ? 1.0f / sqrtf((red[0] + red[1] + red[2] + red[3]) / (float)A.k + 1e-6f) : 1.0f;
    };
    auto write = [&](int i, float4 v, uint2 gw, float inv) {
        float g[4] = {1.0f, 1.0f, 1.0f, 1.0f};
        if (A.norm_w) {
            g[0] = 1.0f + f16_to_f32((uint16_t)(gw.x & 0xffffu)); g[1] = 1.0f + f16_to_f32((uint16_t)(gw.x >> 16));
            g[2] = 1.0f + f16_to_f32((uint16_t)(gw.y & 0xffffu)); g[3] = 1.0f + f16_to_f32((uint16_t)(gw.y >> 16));
        }
        const uint32_t lo = (uint32_t)f32_to_f16(v.x * inv * g[0]) | ((uint32_t)f32_to_f16(v.y * inv * g[1]) << 16);
        const uint32_t hi = (uint32_t)f32_to_f16(v.z * inv * g[2]) | ((uint32_t)f32_to_f16(v.w * inv * g[3]) << 16);
        *reinterpret_cast<uint2*>(out + i) = make_uint2(lo, hi);
    };
    if constexpr (NV > 0) {
        float4 v[NV];
        uint2 gw[NV];
#pragma unroll
        for (int j = 0; j < NV; ++j)
            if (4 * tid + 1024 * j < A.k) v[j] = ld4(x + 4 * tid + 1024 * j);
#pragma unroll
        for (int j = 0; j < NV; ++j)
            if (A.norm_w && 4 * tid + 1024 * j < A.k) gw[j] = *reinterpret_cast<const uint2*>(A.norm_w + 4 * tid + 1024 * j);
#pragma unroll
        for (int j = 0; j < NV; ++j)
            if (4 * tid + 1024 * j < A.k) square(v[j]);
        const float inv = total();
#pragma unroll
        for (int j = 0; j < NV; ++j)
            if (4 * tid + 1024 * j < A.k) write(4 * tid + 1024 * j, v[j], gw[j], inv);
    } else {
        for (int i = 4 * tid; i < A.k; i += 1024) square(ld4(x + i));
        const float inv = total();
        for (int i = 4 * tid; i < A.k; i += 1024)
            write(i, ld4(x + i), A.norm_w ? *reinterpret_cast<const uint2*>(A.norm_w + i) : make_uint2(0, 0), inv);
    }
}
extern "C" __global__ __launch_bounds__(256) void qm_rms_norm_f16(RmsNormArgs A) { rms_norm_f16_body<0>(A); }
extern "C" __global__ __launch_bounds__(256) void qm_rms_norm_f16_k1024(RmsNormArgs A) { rms_norm_f16_body<1>(A); }
extern "C" __global__ __launch_bounds__(256) void qm_rms_norm_f16_k2048(RmsNormArgs A) { rms_norm_f16_body<2>(A); }
extern "C" __global__ __launch_bounds__(256) void qm_rms_norm_f16_k4096(RmsNormArgs A) { rms_norm_f16_body<4>(A); }

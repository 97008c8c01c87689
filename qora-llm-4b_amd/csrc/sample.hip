// sample.hip -- next-token sampling on the device for gfx950: penalties,
// top-k, temperature softmax, top-p and the xorshift64 draw, so that the
// logits never leave HBM (generate.rs:58-82,334-384; the wgpu path's twin,
// gpu_inference.rs:867-931).
//
// qm_sample_penalties (one workgroup): the repetition penalty over the last
// 64 generated ids in order (repeats apply again, as the reference's loop
// does), the presence penalty once per distinct generated id, then an
// optional banned id set to -inf (generate.rs:189-195).
//
// The top k of the reference's stable descending sort (logit desc, index
// asc) without sorting the vocabulary:
//   qm_sample_select: each workgroup finds the first k of its slice of the
//      vocabulary by a radix select over an order-preserving 32-bit key (-0
//      folded onto +0, which compare equal in the reference's sort; NaN
//      below -inf): four 8-bit digits, LDS histograms with integer atomics
//      (order-independent), then every key above the threshold and, of the
//      keys equal to it, the lowest indices (a block scan of the per-thread
//      counts makes that choice deterministic).
//      The slice's candidates are sorted (bitonic, in LDS).
//   qm_sample_top_k (one workgroup of 1024 threads): merge of the slices'
//      sorted lists up to k elements; then the reference's sequential f32
//      arithmetic on one thread: the softmax sum, the top-p cutoff, the
//      total and the cumulative draw, in the reference's order and rounding
//      (contraction off in these kernels).  exp is taken in double and rounded to f32 (the
//      reference calls libm expf, correctly rounded but for rare half-way
//      cases).
// Greedy (temperature <= 0) is the same selection with k = 1.
//
// For k up to 64 and enough slices (the host's rule) a shorter way, two launches:
//   qm_sample_slices: each workgroup applies the penalties to its slice of the
//      vocabulary and writes the slice's largest key;
//   qm_sample_draw (one workgroup): the k-th largest of those keys is a lower
//      bound of the k-th largest logit, and only the k slices with the largest
//      keys hold candidates, so k slices are read instead of sorting each; the
//      candidates that reach the bound are ranked by counting where they are
//      few (logits spread over the vocabulary) and cut down to k by radix
//      select where they are many (large logits beside each other, equal
//      ones, a vocabulary mostly masked), and one wave draws, its lanes
//      holding the probabilities.
// What bounded the longer way was its chain of steps, not bytes: penalties 4.8
// us, select 11.8 (four radix passes, a scan and a sort per slice), merge and
// draw 14.6 (20 rounds of a 64-lane maximum, then one thread's loads from
// LDS); now 4.1 and 11.4 us (248,320 logits, top 20, presence penalty over 1000
// ids).  The whole call in a replayed graph, us, longer / shorter way: spread
// logits 28.8 / 14.5, sorted ones 29.0 / 22.6, all equal 30.3 / 26.8, all but
// five masked 28.6 / 26.8; at top 64 57.3 / 25.4, 58.2 / 45.3, 60.8 / 48.7,
// 55.6 / 48.7; 32,000 generated ids 65.8 / 36.1.
#include "qm_device.h"
#include "qm_kernel_args.h"

#define SMP_THREADS 1024
#define SMP_MAX_K 1024
#define SMP_MAX_CAND 8192          // stage-1 candidates (slices x k), merged in LDS
#define SMP_MAX_LISTS 256          // stage-1 slices (vocabulary / 1024 at most)
#define SMP_MAX_VOCAB 262144       // the presence bitmap in LDS (32 KB)
#define SMP_MAX_SLICE 1024         // logits per workgroup of qm_sample_slices (256, 512 or 1024)
#define SMP_DRAW_CAND 4096         // candidates of qm_sample_draw: k <= 64 threads x 64 logits
// Candidates ranked by counting, a quadratic cost; above, radix select comes
// first.  Whole call, us, counting / select (248,320 logits, top 20): 128
// candidates 15.7 / 16.6, 224 16.5 / 17.6, 320 19.4 / 17.5, 512 24.9 / 17.7,
// 1000 44.8 / 17.9, 4000 453 / 21.0; at top 64 they cross near 192.
#define SMP_COUNT_CAND 256

// Larger logit -> larger key; -0 == +0; NaN below every number.
QM_DEV uint32_t logit_key(float v) {
    uint32_t u = __float_as_uint(v);
    if (v != v) return 0u;
    if (u == 0x80000000u) u = 0u;
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

QM_DEV float key_logit(uint32_t k) {
    return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

extern "C" __global__ __launch_bounds__(SMP_THREADS) void qm_sample_penalties(SampleArgs A) {
#pragma clang fp contract(off)
    __shared__ uint32_t seen[(SMP_MAX_VOCAB + 31) / 32];
    const int tid = threadIdx.x;
    const int n = A.n_generated;
    // generate.rs:58-69
    if (A.repetition_penalty > 1.0f && tid == 0) {
        const int window = min(n, 64);
        for (int i = n - window; i < n; ++i) {
            const int tok = A.generated[i];
            if (tok < 0 || tok >= A.vocab) continue;
            const float l = A.logits[tok];
            A.logits[tok] = l > 0.0f ? __fdiv_rn(l, A.repetition_penalty) : __fmul_rn(l, A.repetition_penalty);
        }
    }
    // generate.rs:72-82: once per distinct id, by the thread whose bit-set
    // in an LDS bitmap of the vocabulary finds the bit clear
    const bool presence = A.presence_penalty > 0.0f && n > 0;
    if (presence)
        for (int i = tid; i < (A.vocab + 31) / 32; i += SMP_THREADS) seen[i] = 0u;
    __syncthreads();
    if (presence) {
        for (int i = tid; i < n; i += SMP_THREADS) {
            const int tok = A.generated[i];
            if (tok < 0 || tok >= A.vocab) continue;
            const uint32_t bit = 1u << (tok & 31);
            if (!(atomicOr(&seen[tok >> 5], bit) & bit)) A.logits[tok] = __fsub_rn(A.logits[tok], A.presence_penalty);
        }
    }
    __syncthreads();
    if (tid == 0 && A.banned >= 0 && A.banned < A.vocab) A.logits[A.banned] = -__builtin_inff();
}

// The penalties and the largest key of one slice [w CH, (w + 1) CH) of the
// vocabulary, in place: the same arithmetic per logit as
// qm_sample_penalties (a logit's penalties depend on no other's).
extern "C" __global__ __launch_bounds__(256) void qm_sample_slices(SampleArgs A) {
#pragma clang fp contract(off)
    __shared__ uint32_t seen[SMP_MAX_SLICE / 32];
    __shared__ uint32_t wmax[4];
    const int tid = threadIdx.x, lane = tid & 63;
    const int s0 = blockIdx.x * A.chunk, s1 = min(s0 + A.chunk, A.vocab);
    const int n = A.n_generated;
    const bool repeat = A.repetition_penalty > 1.0f && n > 0, presence = A.presence_penalty > 0.0f && n > 0;
    if (presence && tid < SMP_MAX_SLICE / 32) seen[tid] = 0u;
    // generate.rs:58-69: lane i holds the i-th id of the window; the first
    // occurrence of an id applies its penalty as often as the id occurs
    if (repeat && tid < 64) {
        const int window = min(n, 64);
        const int tok = lane < window ? A.generated[n - window + lane] : -1;
        int count = 0, first = 64;
        for (int i = 63; i >= 0; --i) {
            const bool same = __builtin_amdgcn_readlane(tok, i) == tok;
            count += same;
            first = same ? i : first;
        }
        if (tok >= s0 && tok < s1 && first == lane) {
            float l = A.logits[tok];
            for (int i = 0; i < count; ++i)
                l = l > 0.0f ? __fdiv_rn(l, A.repetition_penalty) : __fmul_rn(l, A.repetition_penalty);
            A.logits[tok] = l;
        }
    }
    __syncthreads();
    // generate.rs:72-82: once per distinct id
    if (presence)
        for (int i = tid; i < n; i += 256) {
            const int tok = A.generated[i];
            if (tok < s0 || tok >= s1) continue;
            const uint32_t bit = 1u << ((tok - s0) & 31);
            if (!(atomicOr(&seen[(tok - s0) >> 5], bit) & bit)) A.logits[tok] = __fsub_rn(A.logits[tok], A.presence_penalty);
        }
    __syncthreads();
    if (tid == 0 && A.banned >= s0 && A.banned < s1) A.logits[A.banned] = -__builtin_inff();
    __syncthreads();
    uint32_t m = 0;
#pragma unroll
    for (int j = 0; j < SMP_MAX_SLICE / 256; ++j) {
        const int i = s0 + tid + 256 * j;
        if (i < s1) m = max(m, logit_key(A.logits[i]));
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, off));
    if (lane == 0) wmax[tid >> 6] = m;
    __syncthreads();
    if (tid == 0) reinterpret_cast<uint32_t*>(A.cand)[blockIdx.x] = max(max(wmax[0], wmax[1]), max(wmax[2], wmax[3]));
}

// Candidate order: key descending, then index ascending (descending for
// tie_last).  Zero sorts last.
QM_DEV uint64_t cand_pack(uint32_t key, int i, bool tie_last) {
    return ((uint64_t)key << 32) | (tie_last ? (uint32_t)i : 0xffffffffu - (uint32_t)i);
}
QM_DEV int32_t cand_id(uint64_t c, bool tie_last) {
    return tie_last ? (int32_t)(uint32_t)c : (int32_t)(0xffffffffu - (uint32_t)c);
}

// The radix digit of one pass, by wave 0: the largest d with
// sum(hist[e], e > d) + hist[d] >= rank.  Lane l holds bins 4l .. 4l + 3;
// suffix sums over lanes by shuffles.  Writes the digit and the count above
// it to out[0], out[1].
QM_DEV void radix_pick(const uint32_t* hist, uint32_t rank, uint32_t* out) {
    const int l = threadIdx.x;
    uint32_t h[4], s = 0;
#pragma unroll
    for (int b = 0; b < 4; ++b) s += (h[b] = hist[4 * l + b]);
    uint32_t incl = s;                     // sum over lanes >= l
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t v = __shfl_down(incl, off);
        if (l + off < 64) incl += v;
    }
    uint32_t above = incl - s;             // bins of the lanes above this one
    int found = -1;
    uint32_t found_above = 0;
#pragma unroll
    for (int b = 3; b >= 0; --b) {
        if (found < 0 && above + h[b] >= rank) {
            found = 4 * l + b;
            found_above = above;
        }
        above += h[b];
    }
    const uint64_t any = __ballot(found >= 0);
    const int top = 63 - __builtin_clzll(any);   // the highest lane holding the answer
    if (l == top) {
        out[0] = (uint32_t)found;
        out[1] = found_above;
    }
}

// Radix select over the keys logit_key(x[lo .. hi)) of the workgroup's
// threads: the key of the rank0-th largest, and how many keys equal to it
// are within the top rank0.
QM_DEV void radix_select(const float* x, int lo, int hi, uint32_t rank0, uint32_t* hist, uint32_t* pick,
                         uint32_t& prefix, uint32_t& rank) {
    const int tid = threadIdx.x;
    uint32_t mask = 0;
    prefix = 0;
    rank = rank0;
    for (int shift = 24; shift >= 0; shift -= 8) {
        for (int i = tid; i < 256; i += blockDim.x) hist[i] = 0;
        __syncthreads();
        for (int i = lo; i < hi; ++i) {
            const uint32_t key = logit_key(x[i]);
            if ((key & mask) == prefix) atomicAdd(&hist[(key >> shift) & 255u], 1u);
        }
        __syncthreads();
        if (tid < 64) radix_pick(hist, rank, pick);
        __syncthreads();
        prefix |= pick[0] << shift;
        rank -= pick[1];
        mask |= 255u << shift;
        __syncthreads();
    }
}

// In-place bitonic sort of c[0 .. P) (P a power of two), descending.
QM_DEV void bitonic_desc(uint64_t* c, int P) {
    for (int size = 2; size <= P; size <<= 1) {
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            for (int i = threadIdx.x; i < P; i += blockDim.x) {
                const int j = i ^ stride;
                if (j > i) {
                    const bool desc = (i & size) == 0;
                    const uint64_t a = c[i], b = c[j];
                    if (desc ? a < b : a > b) {
                        c[i] = b;
                        c[j] = a;
                    }
                }
            }
            __syncthreads();
        }
    }
}

// Stage 1: workgroup w (256 threads) takes the slice [w CH, (w + 1) CH) of
// the vocabulary, thread t the contiguous elements t * per .. + per - 1 of
// it, and writes the slice's first min(k, slice length) elements of the
// global order, sorted, to cand[w k ..] (zeros after them).  Every element
// of the global top k is among its slice's top k.
extern "C" __global__ __launch_bounds__(256) void qm_sample_select(SampleArgs A) {
    __shared__ uint32_t hist[256];
    __shared__ uint32_t scan[256];
    __shared__ uint32_t pick[2], ncand;
    __shared__ uint64_t loc[SMP_MAX_K];
    const int tid = threadIdx.x, w = blockIdx.x;
    const int V = A.vocab;
    const bool greedy = !(A.temperature > 0.0f);
    const int k = greedy ? 1 : min(A.top_k, V);
    const bool tie_last = greedy && (A.flags & QMK_SAMPLE_WGPU);
    const int per = A.chunk / 256;
    const int s0 = w * A.chunk, s1 = min(s0 + A.chunk, V);
    const int lo = min(s0 + tid * per, s1), hi = min(lo + per, s1);
    const int kk = min(k, s1 - s0);

    uint32_t prefix, rank;
    radix_select(A.logits, lo, hi, (uint32_t)kk, hist, pick, prefix, rank);
    // keys above the threshold, then `rank` of the equal keys in index order
    // (reversed for tie_last), ranked by a block scan of per-thread counts
    uint32_t eq = 0;
    for (int i = lo; i < hi; ++i) eq += logit_key(A.logits[i]) == prefix;
    scan[tid] = eq;
    if (tid == 0) ncand = 0;
    __syncthreads();
    for (int off = 1; off < 256; off <<= 1) {
        const uint32_t v = tid >= off ? scan[tid - off] : 0u;
        __syncthreads();
        scan[tid] += v;
        __syncthreads();
    }
    uint32_t before = tie_last ? scan[255] - scan[tid] : scan[tid] - eq;
    for (int j = 0; j < hi - lo; ++j) {
        const int i = tie_last ? hi - 1 - j : lo + j;
        const uint32_t key = logit_key(A.logits[i]);
        bool take = key > prefix;
        if (key == prefix) take = before++ < rank;
        if (take) {
            const uint32_t slot = atomicAdd(&ncand, 1u);
            if (slot < (uint32_t)kk) loc[slot] = cand_pack(key, i, tie_last);
        }
    }
    int P = 1;
    while (P < k) P <<= 1;
    __syncthreads();
    for (int i = kk + tid; i < P; i += 256) loc[i] = 0;
    __syncthreads();
    bitonic_desc(loc, P);
    uint64_t* out = A.cand + (size_t)w * k;
    for (int i = tid; i < k; i += 256) out[i] = loc[i];
}

// Stage 2 (one workgroup): merge the slices' sorted lists into the first k
// of the global order (wave 0 repeatedly takes the largest list head), and
// draw.
extern "C" __global__ __launch_bounds__(SMP_THREADS) void qm_sample_top_k(SampleArgs A) {
#pragma clang fp contract(off)
    __shared__ uint64_t cand[SMP_MAX_CAND];
    __shared__ uint64_t top[SMP_MAX_K];
    __shared__ float prob[SMP_MAX_K];
    __shared__ float sh_sum;

    const int tid = threadIdx.x;
    const int V = A.vocab;
    const bool greedy = !(A.temperature > 0.0f);
    const int k = greedy ? 1 : min(A.top_k, V);
    const bool tie_last = greedy && (A.flags & QMK_SAMPLE_WGPU);
    const int n = A.n_cand, nl = n / k;    // lists of k
    for (int i = tid; i < n; i += SMP_THREADS) cand[i] = A.cand[i];
    __syncthreads();
    if (tid < 64) {
        // lane l owns lists l, l + 64, ... (at most SMP_MAX_LISTS / 64)
        int head[SMP_MAX_LISTS / 64];
        uint64_t hv[SMP_MAX_LISTS / 64];     // current head values; 0 when exhausted
#pragma unroll
        for (int j = 0; j < SMP_MAX_LISTS / 64; ++j) {
            const int list = tid + 64 * j;
            head[j] = 0;
            hv[j] = list < nl ? cand[list * k] : 0;
        }
        for (int r = 0; r < k; ++r) {
            uint64_t best = hv[0];
            int best_j = 0;
#pragma unroll
            for (int j = 1; j < SMP_MAX_LISTS / 64; ++j)
                if (hv[j] > best) {
                    best = hv[j];
                    best_j = j;
                }
            uint64_t m = best;
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) {
                const uint64_t o = __shfl_xor(m, off);
                m = o > m ? o : m;
            }
            // non-zero composites are distinct; the lowest lane holding the
            // maximum advances that list
            const uint64_t holders = __ballot(best == m);
            if (tid == __builtin_ctzll(holders)) {
#pragma unroll
                for (int j = 0; j < SMP_MAX_LISTS / 64; ++j)
                    if (j == best_j) {
                        const int list = tid + 64 * j;
                        head[j]++;
                        hv[j] = head[j] < k ? cand[list * k + head[j]] : 0;
                    }
            }
            if (tid == 0) top[r] = m;
        }
    }
    __syncthreads();
    if (A.top_ids && tid < k) A.top_ids[tid] = cand_id(top[tid], tie_last);
    if (greedy) {                      // generate.rs:335-342 (first maximum; last for the wgpu twin)
        if (tid == 0) A.token_out[0] = cand_id(top[0], tie_last);
        return;
    }

    // generate.rs:345-383 (the wgpu twin, gpu_inference.rs:874-905,
    // divides by the sum instead of multiplying by its inverse and has no
    // zero-sum exits)
    const float inv_temp = __fdiv_rn(1.0f, A.temperature);
    const float max_logit = key_logit((uint32_t)(top[0] >> 32));
    if (tid < k) {
        const float l = key_logit((uint32_t)(top[tid] >> 32));
        prob[tid] = (float)exp((double)__fmul_rn(__fsub_rn(l, max_logit), inv_temp));
    }
    __syncthreads();
    if (tid == 0) {
        float sum = 0.0f;
        for (int i = 0; i < k; ++i) sum = __fadd_rn(sum, prob[i]);
        sh_sum = sum;
    }
    __syncthreads();
    const float sum = sh_sum;
    const bool wgpu = A.flags & QMK_SAMPLE_WGPU;
    if (!wgpu && sum <= 0.0f) {
        if (tid == 0) A.token_out[0] = cand_id(top[0], false);
        return;
    }
    if (tid < k) prob[tid] = wgpu ? __fdiv_rn(prob[tid], sum) : __fmul_rn(prob[tid], __fdiv_rn(1.0f, sum));
    __syncthreads();
    if (A.top_probs && tid < k) A.top_probs[tid] = prob[tid];
    if (tid != 0) return;
    float cumsum = 0.0f;
    int cutoff = k;
    for (int i = 0; i < k; ++i) {
        cumsum = __fadd_rn(cumsum, prob[i]);
        if (cumsum >= A.top_p) {
            cutoff = i + 1;
            break;
        }
    }
    float total = 0.0f;
    for (int i = 0; i < cutoff; ++i) total = __fadd_rn(total, prob[i]);
    if (!wgpu && total <= 0.0f) {
        A.token_out[0] = cand_id(top[0], false);
        return;
    }
    // Rng::next_f32, generate.rs:46-54
    uint64_t s = A.rng_state[0];
    s ^= s << 13;
    s ^= s >> 7;
    s ^= s << 17;
    A.rng_state[0] = s;
    const float rand_val = __fmul_rn((float)(uint32_t)(s >> 40) / 16777216.0f, total);
    float accum = 0.0f;
    int32_t tok = cand_id(top[0], false);
    for (int i = 0; i < cutoff; ++i) {
        accum = __fadd_rn(accum, prob[i]);
        if (accum >= rand_val) {
            tok = cand_id(top[i], false);
            break;
        }
    }
    A.token_out[0] = tok;
}

// The composites (key, index) of the logits of `m` slices, in any order:
// f(composite) for each, over all threads.  Eight loads at a time are in
// flight per thread (one after the other, 20 slices took 10 us).
template <class F>
QM_DEV void for_slices(const SampleArgs& A, const int* list, int m, bool tie_last, F f) {
    const int shift = 31 - __builtin_clz(A.chunk), total = m << shift;   // chunk is a power of two
    for (int i0 = threadIdx.x; i0 < total; i0 += 8 * SMP_THREADS) {
        int id[8];
        float l[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int i = min(i0 + u * SMP_THREADS, total - 1);
            id[u] = (list[i >> shift] << shift) + (i & (A.chunk - 1));
            l[u] = A.logits[min(id[u], A.vocab - 1)];
            if (i0 + u * SMP_THREADS >= total) id[u] = A.vocab;
        }
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (id[u] < A.vocab) f(cand_pack(logit_key(l[u]), id[u], tie_last));
    }
}

// The k-th largest of the n distinct composites in LDS, by radix select of
// eight-bit digits from the top, ended as soon as a digit's bin is taken
// whole: exactly k of them are >= the value returned.  All threads call it.
QM_DEV uint64_t kth_largest(const uint64_t* c, int n, int k, uint32_t* hist, uint32_t* pick) {
    const int tid = threadIdx.x, lane = tid & 63;
    uint64_t prefix = 0, mask = 0;
    uint32_t rank = (uint32_t)k;
    for (int shift = 56; shift >= 0; shift -= 8) {
        __syncthreads();
        if (tid < 256) hist[tid] = 0;
        __syncthreads();
        for (int i = tid; i < n; i += SMP_THREADS) {
            const uint64_t v = c[i];
            if ((v & mask) != prefix) continue;
            const uint32_t d = (uint32_t)(v >> shift) & 255u;
            // near logits share their upper digits: one add per wave then
            const uint64_t on = __ballot(1);
            if (__ballot(d == (uint32_t)__builtin_amdgcn_readfirstlane((int)d)) == on) {
                if (lane == __builtin_ctzll(on)) atomicAdd(&hist[d], (uint32_t)__popcll(on));
            } else {
                atomicAdd(&hist[d], 1u);
            }
        }
        __syncthreads();
        if (tid < 64) radix_pick(hist, rank, pick);
        __syncthreads();
        prefix |= (uint64_t)pick[0] << shift;
        rank -= pick[1];
        mask |= 255ull << shift;
        if (hist[pick[0]] == rank) break;
    }
    return prefix;
}

// The selection over qm_sample_slices' keys, and the draw, for k <= 64 and
// at least k slices (see the head of this file).
extern "C" __global__ __launch_bounds__(SMP_THREADS) void qm_sample_draw(SampleArgs A) {
#pragma clang fp contract(off)
    __shared__ __attribute__((aligned(16))) uint32_t smax[SMP_MAX_LISTS];
    __shared__ int list[64];
    __shared__ uint64_t cand[SMP_DRAW_CAND];
    __shared__ uint64_t tmax[SMP_THREADS];
    __shared__ uint64_t top[64];
    __shared__ uint32_t hist[256], pick[2];
    __shared__ uint32_t bound, ncand;
    const int tid = threadIdx.x, lane = tid & 63;
    const bool greedy = !(A.temperature > 0.0f);
    const int k = greedy ? 1 : min(A.top_k, A.vocab);
    const bool tie_last = greedy && (A.flags & QMK_SAMPLE_WGPU);
    const int ns = (A.vocab + A.chunk - 1) / A.chunk;
    // the generator's state is needed last and requested first
    const uint64_t rng = tid < 64 && !greedy ? A.rng_state[0] : 0;
    // slices in the order that ties are taken in
    if (tid < SMP_MAX_LISTS)
        smax[tid] = tid < ns ? reinterpret_cast<const uint32_t*>(A.cand)[tie_last ? ns - 1 - tid : tid] : 0u;
    if (tid == 0) ncand = 0;
    __syncthreads();
    // The first k slices by (maximum, order): the k-th one's maximum is a key
    // that at least k logits reach, and a logit of any other slice comes
    // after those k (equal ones stand in an earlier slice).  Four threads per
    // slice count the slices before it.
    {
        const int i = tid >> 2;
        const uint32_t mine = smax[i];
        int above = 0;
#pragma unroll 4
        for (int j = 4 * (tid & 3); j < SMP_MAX_LISTS; j += 16) {   // zeros past ns
            const uint4 o = *reinterpret_cast<const uint4*>(&smax[j]);
            above += (o.x > mine || (o.x == mine && j < i)) + (o.y > mine || (o.y == mine && j + 1 < i)) +
                     (o.z > mine || (o.z == mine && j + 2 < i)) + (o.w > mine || (o.w == mine && j + 3 < i));
        }
        above += __shfl_xor(above, 1);
        above += __shfl_xor(above, 2);
        if (i < ns && (tid & 3) == 0 && above < k) {
            list[above] = tie_last ? ns - 1 - i : i;
            if (above == k - 1) bound = mine;
        }
    }
    __syncthreads();
    // at most 64 logits a thread
    uint64_t m = 0;                        // the thread's largest
    auto collect = [&](uint64_t from) {
        for_slices(A, list, k, tie_last, [&](uint64_t c) {
            if (c < from) return;
            m = c > m ? c : m;
            const uint32_t slot = atomicAdd(&ncand, 1u);
            if (slot < SMP_DRAW_CAND) cand[slot] = c;
        });
        __syncthreads();
        return (int)ncand;
    };
    int n = collect((uint64_t)bound << 32);
    if (k == 1 && n > SMP_COUNT_CAND) {     // the largest is among the threads' largest
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            const uint64_t o = __shfl_xor(m, off);
            m = o > m ? o : m;
        }
        if (lane == 0) tmax[tid >> 6] = m;
        __syncthreads();
        for (int w = 0; w < SMP_THREADS / 64; ++w) m = tmax[w] > m ? tmax[w] : m;
        if (tid == 0) cand[0] = m;
        __syncthreads();
        n = 1;
    }
    if (n > SMP_DRAW_CAND) {
        // Large logits beside each other, or equal ones: the k-th largest of
        // the threads' maxima is a closer bound, reached in exactly k
        // threads, so by at most 64 k logits.
        tmax[tid] = m;
        const uint64_t from = kth_largest(tmax, SMP_THREADS, k, hist, pick);
        if (tid == 0) ncand = 0;
        __syncthreads();
        n = collect(from);
    }
    if (n > SMP_COUNT_CAND) {
        const uint64_t from = kth_largest(cand, n, k, hist, pick);
        uint64_t own[SMP_DRAW_CAND / SMP_THREADS];
#pragma unroll
        for (int j = 0; j < SMP_DRAW_CAND / SMP_THREADS; ++j) {
            const int i = tid + j * SMP_THREADS;
            own[j] = i < n ? cand[i] : 0;
        }
        __syncthreads();
        if (tid == 0) ncand = 0;
        __syncthreads();
#pragma unroll
        for (int j = 0; j < SMP_DRAW_CAND / SMP_THREADS; ++j)
            if (tid + j * SMP_THREADS < n && own[j] >= from) cand[atomicAdd(&ncand, 1u)] = own[j];
        __syncthreads();
        n = k;
    }
    // rank by counting, eight threads per candidate
    for (int i0 = 0; i0 < n; i0 += SMP_THREADS / 8) {
        const int i = i0 + (tid >> 3);
        const uint64_t mine = cand[min(i, n - 1)];
        int above = 0;
#pragma unroll 4
        for (int j = tid & 7; j < n; j += 8) above += cand[j] > mine;
        above += __shfl_xor(above, 1);
        above += __shfl_xor(above, 2);
        above += __shfl_xor(above, 4);
        if (i < n && (tid & 7) == 0 && above < k) top[above] = mine;
    }
    __syncthreads();
    if (tid >= 64) return;
    const uint64_t c = lane < k ? top[lane] : 0;
    const int32_t id = cand_id(c, tie_last), best = __builtin_amdgcn_readlane(id, 0);
    if (A.top_ids && lane < k) A.top_ids[lane] = id;
    if (greedy) {                      // generate.rs:335-342 (first maximum; last for the wgpu twin)
        if (lane == 0) A.token_out[0] = best;
        return;
    }
    // generate.rs:345-383 as in qm_sample_top_k, in the reference's order
    // and rounding.  Its cutoff, total and draw loops all add the same
    // probabilities from zero: one running sum, lane i keeping the i-th.
    const float inv_temp = __fdiv_rn(1.0f, A.temperature);
    const float l = key_logit((uint32_t)(c >> 32));
    float p = (float)exp((double)__fmul_rn(__fsub_rn(l, readlane_f32(l, 0)), inv_temp));
    float sum = 0.0f;
    for (int i = 0; i < k; ++i) sum = __fadd_rn(sum, readlane_f32(p, i));
    const bool wgpu = A.flags & QMK_SAMPLE_WGPU;
    if (!wgpu && sum <= 0.0f) {
        if (lane == 0) A.token_out[0] = best;
        return;
    }
    p = wgpu ? __fdiv_rn(p, sum) : __fmul_rn(p, __fdiv_rn(1.0f, sum));
    if (A.top_probs && lane < k) A.top_probs[lane] = p;
    float run = 0.0f, upto = 0.0f;
    for (int i = 0; i < k; ++i) {
        run = __fadd_rn(run, readlane_f32(p, i));
        upto = lane == i ? run : upto;
    }
    const uint64_t reach = __ballot(lane < k && upto >= A.top_p);
    const int cutoff = reach ? __builtin_ctzll(reach) + 1 : k;
    const float total = readlane_f32(upto, cutoff - 1);
    if (!wgpu && total <= 0.0f) {
        if (lane == 0) A.token_out[0] = best;
        return;
    }
    // Rng::next_f32, generate.rs:46-54
    uint64_t s = rng;
    s ^= s << 13;
    s ^= s >> 7;
    s ^= s << 17;
    const float rand_val = __fmul_rn((float)(uint32_t)(s >> 40) / 16777216.0f, total);
    const uint64_t hit = __ballot(lane < cutoff && upto >= rand_val);
    const int32_t tok = hit ? __builtin_amdgcn_readlane(id, __builtin_ctzll(hit)) : best;
    if (lane == 0) {
        A.rng_state[0] = s;
        A.token_out[0] = tok;
    }
}

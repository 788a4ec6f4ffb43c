// The Mamba-2 mixer between its two projections: short causal convolution with SiLU over x, B and C (short_conv.hip), the
// state-space recurrence per head, and the gated grouped RMS norm. Everything here is f32 in both arithmetics; only the rows that
// leave for the output projection take the arithmetic's activation type.
#include "stack_dev.hpp"

namespace rk {

namespace {

constexpr int kScanP = 64;            // columns of the state one workgroup holds
constexpr int kScanTokens = 8;        // tokens staged at once

// The recurrence token by token, of runs of fewer than `below` tokens: thread (p, q) holds the state of column p for rows q,
// q + 4, ...
template <int NPT>
__global__ __launch_bounds__(256) void k_mamba_scan(MambaJob j, int below) {
    extern __shared__ float sm[];
    const MambaShape sh = j.sh;
    const int N = sh.state, P = sh.vdim, C = sh.channels();
    const int h = blockIdx.x, g = h / (sh.heads / sh.groups);
    const int p = blockIdx.y * kScanP + (threadIdx.x & 63), q = threadIdx.x >> 6;
    const SeqRun run = j.runs.runs[blockIdx.z];
    if (run.n >= below) return;
    float * sB = sm, * sC = sB + kScanTokens * N, * part = sC + kScanTokens * N;      // part [tokens][4][64]
    __shared__ float s_dt[kScanTokens], s_decay[kScanTokens];
    const bool mine = p < P;
    float * st = j.state + (((size_t)run.slot * sh.heads + h) * N) * P + p;
    float S[NPT];
#pragma unroll
    for (int i = 0; i < NPT; ++i) {
        const int n = q + 4 * i;
        S[i] = (mine && n < N && !(run.flags & 1)) ? st[(size_t)n * P] : 0.0f;
    }
    const float a = expf(j.A_log[h]), D = j.D[h], bias = j.dt_bias[h];
    for (int base = 0; base < run.n; base += kScanTokens) {
        const int cnt = min(kScanTokens, run.n - base);
        __syncthreads();
        for (int i = threadIdx.x; i < cnt * N; i += 256) {
            const int tk = i / N, n = i % N;
            const float * row = j.xbc + (size_t)j.runs.tok[run.start + base + tk] * C + sh.inner() + g * N + n;
            sB[i] = row[0];
            sC[i] = row[(size_t)sh.groups * N];
        }
        if ((int)threadIdx.x < cnt) {
            const float dt = softplus_f(j.proj[(size_t)j.runs.tok[run.start + base + threadIdx.x] * j.ld + sh.inner() + C + h] + bias);
            s_dt[threadIdx.x] = dt;
            s_decay[threadIdx.x] = expf(-a * dt);
        }
        __syncthreads();
        for (int tk = 0; tk < cnt; ++tk) {
            const float x = mine ? j.xbc[(size_t)j.runs.tok[run.start + base + tk] * C + h * P + p] : 0.0f;
            const float dx = s_dt[tk] * x, dec = s_decay[tk];
            float y = 0.0f;
#pragma unroll
            for (int i = 0; i < NPT; ++i) {
                const int n = q + 4 * i;
                if (n < N) {
                    S[i] = S[i] * dec + sB[tk * N + n] * dx;
                    y += S[i] * sC[tk * N + n];
                }
            }
            part[(tk * 4 + q) * 64 + (threadIdx.x & 63)] = y;
        }
        __syncthreads();
        for (int tk = q; tk < cnt; tk += 4) {
            if (!mine) continue;
            float y = 0.0f;
#pragma unroll
            for (int i = 0; i < 4; ++i) y += part[(tk * 4 + i) * 64 + (threadIdx.x & 63)];
            const int t = j.runs.tok[run.start + base + tk];
            j.y[(size_t)t * sh.inner() + h * P + p] = y + D * j.xbc[(size_t)t * C + h * P + p];
        }
    }
#pragma unroll
    for (int i = 0; i < NPT; ++i) {
        const int n = q + 4 * i;
        if (mine && n < N) st[(size_t)n * P] = S[i];
    }
}

constexpr int kChunk = 64;            // tokens of a chunk
constexpr int kChunkP = 64;           // state columns of a workgroup
constexpr int kChunkN = 128;          // most state rows of the chunked kernels
constexpr int kWalkP = 32;            // of a workgroup that walks the chunks of a run
constexpr int kChunkLeast = 32;       // tokens of a run that goes by chunks
constexpr int kWalkMost = 128;        // tokens of the longest run up to which a step's runs are walked: four layers of a
                                      // prompt of 32 tokens take 45 us less than by three launches, of 128 15 us, of 160 21 us more
constexpr int kLdX = kChunkP + 4;     // a step of 4 rows is 16 LDS banks: the four lane groups of an operand do not meet

// The recurrence in chunks of 64 tokens on the f32 matrix instruction. With l_t the running sum of -exp(A_log) dt in a
// chunk (kept in double: differences of it are what is exponentiated) and S the state before the chunk,
//   y_t = exp(l_t) S^T C_t + sum over s <= t of exp(l_t - l_s) dt_s (C_t . B_s) x_s + D x_t,
//   S  <- exp(l_last) S + sum over s of exp(l_last - l_s) dt_s B_s x_s^T.
// Longer runs, three launches: what every chunk adds to the state, all chunks at once; the states before the chunks from those sums,
// element by element along a run; the read-outs, all chunks at once. What bounds them is the state of every chunk in memory
// (written, read, written and read: four times 4 N P bytes per head and chunk) and, in the read-outs, the matrix instruction;
// a walk is a chain of 12 to 17 us per chunk whatever the number of runs. 64 heads of 128 x 64, 3321 tokens in five runs: 200
// us, by the walk 321. Tokens past the run's end count as dt = 0, which leaves everything unchanged. VEC: rows can be read
// four columns at a time.

// Chunk c of the step: the chunks of run r are numbered from start / 64 + r, so that the grid needs no list.
__device__ bool chunk_of(const SeqRuns & runs, int c, SeqRun & run, int & base) {
    const int lane = threadIdx.x & 63;
    int r = 0;
    for (int r0 = 0; r0 < runs.n; r0 += 64) {
        const uint64_t before = __ballot(r0 + lane < runs.n && runs.runs[min(r0 + lane, runs.n - 1)].start / kChunk + r0 + lane <= c);
        if (before == 0) break;
        r = r0 + 63 - __clzll((long long)before);
    }
    r = __builtin_amdgcn_readfirstlane(r);
    run = runs.runs[r];
    base = (c - (run.start / kChunk + r)) * kChunk;
    return run.n >= kChunkLeast && base < run.n;
}
// Where the state of a run's chunk lies: a run of at least 32 tokens has no more chunks than pairs of 16 tokens.
__device__ inline size_t chunk_slot(const SeqRun & run, int base) { return (size_t)(run.start / kChunkLeast + base / kChunk); }
// Workgroup x runs on XCD x % 8: the heads of a group share its rows of B and C in one L2.
__device__ inline int chunk_head(int x, int heads) { return heads % 8 == 0 ? (x & 7) * (heads / 8) + (x >> 3) : x; }

struct ChunkSteps {
    double l[kChunk];
    float dt[kChunk];
    int tok[kChunk];
};
__device__ inline int chunk_token(const MambaJob & j, const SeqRun & run, int base, int tk) {
    return j.runs.tok[run.start + min(base + tk, run.n - 1)];
}
// The chunk's tokens, time steps and running decays, by the first wave.
__device__ void chunk_steps(const MambaJob & j, const SeqRun & run, int base, int h, ChunkSteps & st) {
    const int lane = threadIdx.x & 63;
    const int tok = chunk_token(j, run, base, lane);
    const float raw = j.proj[(size_t)tok * j.ld + j.sh.inner() + j.sh.channels() + h];
    const float dt = base + lane < run.n ? softplus_f(raw + j.dt_bias[h]) : 0.0f;
    double l = -(double)expf(j.A_log[h]) * (double)dt;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const double up = __shfl_up(l, o, 64);
        if (lane >= o) l += up;
    }
    st.l[lane] = l;
    st.dt[lane] = dt;
    st.tok[lane] = tok;
}

// Rows of a chunk, `width` columns (a multiple of four for VEC) from column `col`, to LDS rows of ld floats, zero past the
// width up to `padded` (a power of two of at most 128, or at most 128 in all) and past the run's end. In two halves, so that
// everything a workgroup needs is on its way at once.
template <bool VEC, int MOST> struct ChunkRows {
    static constexpr int NV = kChunk * MOST / 4 / 256, LANES = MOST / 4;      // per thread, threads per row
    f4 v[VEC ? NV : 1];
    __device__ void fetch(const MambaJob & j, const SeqRun & run, int base, int col, int width) {
        if constexpr (VEC) {
#pragma unroll
            for (int i = 0; i < NV; ++i) {
                const int tk = threadIdx.x / LANES + 256 / LANES * i, n = 4 * (threadIdx.x % LANES);
                v[i] = *(const f4 *)(j.xbc + (size_t)chunk_token(j, run, base, tk) * j.sh.channels() + col + min(n, width - 4));
            }
        }
    }
    __device__ void store(const MambaJob & j, const SeqRun & run, int base, int col, int width, int padded, float * lds, int ld) const {
        const int cnt = min(kChunk, run.n - base);
        if constexpr (VEC) {
            const int n = 4 * (threadIdx.x % LANES);
            if (n < padded) {
#pragma unroll
                for (int i = 0; i < NV; ++i) {
                    const int tk = threadIdx.x / LANES + 256 / LANES * i;
                    *(f4 *)(lds + tk * ld + n) = n < width && tk < cnt ? v[i] : (f4){0, 0, 0, 0};
                }
            }
        } else {
            for (int i = threadIdx.x; i < kChunk * padded; i += 256) {
                const int tk = i / padded, n = i - tk * padded;
                lds[tk * ld + n] = n < width && tk < cnt ? j.xbc[(size_t)chunk_token(j, run, base, tk) * j.sh.channels() + col + n] : 0.0f;
            }
        }
    }
};

// What a chunk adds to the state, into the chunk's place: wave w makes row tiles w and w + 4. The MFMA's inner index runs over
// tokens 16 k + 4 (lane / 16) + e, so that the rows of an operand lie 4 LDS rows apart.
template <bool VEC>
__global__ __launch_bounds__(256) void k_mamba_chunk_sums(MambaJob j) {
    extern __shared__ __attribute__((aligned(16))) float sm[];
    __shared__ ChunkSteps steps;
    __shared__ float s_w[kChunk];
    const MambaShape sh = j.sh;
    const int N = sh.state, Np = (N + 15) / 16 * 16, P = sh.vdim, LB = Np + 4;
    const int h = chunk_head(blockIdx.x, sh.heads), g = h / (sh.heads / sh.groups), p0 = blockIdx.y * kChunkP;
    SeqRun run;
    int base;
    if (!chunk_of(j.runs, blockIdx.z, run, base)) return;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, r16 = lane & 15, kg = lane >> 4;
    float * sB = sm, * sX = sB + kChunk * LB;
    const int b_col = sh.inner() + g * N, x_col = h * P + p0, x_width = min(P - p0, kChunkP);
    ChunkRows<VEC, kChunkN> rB;
    ChunkRows<VEC, kChunkP> rX;
    rB.fetch(j, run, base, b_col, N);
    rX.fetch(j, run, base, x_col, x_width);
    if (w == 0) {
        chunk_steps(j, run, base, h, steps);
        const double all = __shfl(steps.l[lane], 63, 64);
        s_w[lane] = expf((float)(all - steps.l[lane])) * steps.dt[lane];
        if (lane == 0 && blockIdx.y == 0) j.chunk_decay[chunk_slot(run, base) * sh.heads + h] = expf((float)all);
    }
    rB.store(j, run, base, b_col, N, Np, sB, LB);
    rX.store(j, run, base, x_col, x_width, kChunkP, sX, kLdX);
    __syncthreads();
    float wt[kChunk / 4];
#pragma unroll
    for (int k = 0; k < kChunk / 16; ++k)
#pragma unroll
        for (int e = 0; e < 4; ++e) wt[4 * k + e] = s_w[16 * k + 4 * kg + e];
    float * out = j.chunks + ((chunk_slot(run, base) * sh.heads + h) * N) * P + p0;
    for (int nt = w; nt < Np / 16; nt += 4) {
        f4 d[kChunkP / 16];
#pragma unroll
        for (int c = 0; c < kChunkP / 16; ++c) d[c] = (f4){0, 0, 0, 0};
#pragma unroll
        for (int k = 0; k < kChunk / 16; ++k)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int s = 16 * k + 4 * kg + e;
                const float b = sB[s * LB + 16 * nt + r16] * wt[4 * k + e];
#pragma unroll
                for (int c = 0; c < kChunkP / 16; ++c) d[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(b, sX[s * kLdX + 16 * c + r16], d[c], 0, 0, 0);
            }
#pragma unroll
        for (int c = 0; c < kChunkP / 16; ++c)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int n = 16 * nt + 4 * kg + i, p = 16 * c + r16;
                if (n < N && p < x_width) out[(size_t)n * P + p] = d[c][i];
            }
    }
}

// The states before the chunks in place of what the chunks add, and the state after the run: thread by thread four (VEC) or
// one element of a head's state along the run, four chunks' loads in flight.
template <bool VEC>
__global__ __launch_bounds__(256) void k_mamba_chunk_states(MambaJob j) {
    using V = std::conditional_t<VEC, f4, float>;
    constexpr int W = VEC ? 4 : 1;
    const MambaShape sh = j.sh;
    const SeqRun run = j.runs.runs[blockIdx.z];
    const int h = blockIdx.y, per = sh.state * sh.vdim, at = (blockIdx.x * 256 + threadIdx.x) * W;
    if (run.n < kChunkLeast || at >= per) return;
    const int n_chunks = (run.n + kChunk - 1) / kChunk;
    float * st = j.state + ((size_t)run.slot * sh.heads + h) * per + at;
    const size_t step = (size_t)sh.heads * per;
    float * ch = j.chunks + chunk_slot(run, 0) * step + (size_t)h * per + at;
    const float * decay = j.chunk_decay + chunk_slot(run, 0) * sh.heads + h;
    V S = V{};
    if (!(run.flags & 1)) S = *(const V *)st;
    for (int c = 0; c < n_chunks; c += 4) {
        V add[4];
        float d[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int cc = min(c + u, n_chunks - 1);
            add[u] = *(const V *)(ch + cc * step);
            d[u] = decay[(size_t)cc * sh.heads];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if (c + u >= n_chunks) break;
            *(V *)(ch + (c + u) * step) = S;
            S = S * d[u] + add[u];
        }
    }
    *(V *)st = S;
}

// The read-outs of a chunk: wave w owns token tile w. The decayed products of C and B are made with the tokens s as rows, which
// leaves them where the next product takes its left operand from; C comes from memory in operand order; the state takes B's
// place in LDS once the waves are done with it (three workgroups per CU, one with a place for each).
template <bool VEC>
__global__ __launch_bounds__(256, 3) void k_mamba_chunk_out(MambaJob j) {
    extern __shared__ __attribute__((aligned(16))) float sm[];
    __shared__ ChunkSteps steps;
    const MambaShape sh = j.sh;
    const int N = sh.state, Np = (N + 15) / 16 * 16, P = sh.vdim, C = sh.channels(), LB = Np + 4;
    const int h = chunk_head(blockIdx.x, sh.heads), g = h / (sh.heads / sh.groups), p0 = blockIdx.y * kChunkP;
    SeqRun run;
    int base;
    if (!chunk_of(j.runs, blockIdx.z, run, base)) return;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, r16 = lane & 15, kg = lane >> 4, t0 = 16 * w;
    float * sX = sm, * sB = sX + kChunk * kLdX, * sS = sB;
    const int b_col = sh.inner() + g * N, x_col = h * P + p0, x_width = min(P - p0, kChunkP);
    const int cnt = min(kChunk, run.n - base);
    ChunkRows<VEC, kChunkN> rB;
    ChunkRows<VEC, kChunkP> rX;
    rB.fetch(j, run, base, b_col, N);
    rX.fetch(j, run, base, x_col, x_width);
    f4 ct[kChunkN / 16];                     // C of token t0 + r16, columns 16 k + 4 kg ..
    {
        const float * row = j.xbc + (size_t)chunk_token(j, run, base, t0 + r16) * C + b_col + (size_t)sh.groups * N;
        const bool in = t0 + r16 < cnt;
#pragma unroll
        for (int k = 0; k < kChunkN / 16; ++k) {
            const int n = 16 * k + 4 * kg;
            ct[k] = (f4){0, 0, 0, 0};
            if constexpr (VEC) {
                if (in && n < N) ct[k] = *(const f4 *)(row + n);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) if (in && n + e < N) ct[k][e] = row[n + e];
            }
        }
    }
    const float * st = j.chunks + ((chunk_slot(run, base) * sh.heads + h) * N) * P + p0;
    constexpr int NS = kChunkN * kChunkP / 4 / 256;
    f4 rS[VEC ? NS : 1];
    if constexpr (VEC) {
#pragma unroll
        for (int i = 0; i < NS; ++i) {
            const int n = (threadIdx.x >> 4) + 16 * i, p = 4 * (threadIdx.x & 15);
            rS[i] = *(const f4 *)(st + (size_t)min(n, N - 1) * P + min(p, x_width - 4));
        }
    }
    if (w == 0) chunk_steps(j, run, base, h, steps);
    rB.store(j, run, base, b_col, N, Np, sB, LB);
    rX.store(j, run, base, x_col, x_width, kChunkP, sX, kLdX);
    __syncthreads();
    f4 m[kChunk / 16];                       // of token t0 + r16 with tokens 16 q + 4 kg ..
    {
        const double lt = steps.l[t0 + r16];
#pragma unroll
        for (int q = 0; q < kChunk / 16; ++q) {
            m[q] = (f4){0, 0, 0, 0};
            if (q > w) continue;
            f4 d = {0, 0, 0, 0};
            const float * rb = sB + (16 * q + r16) * LB + 4 * kg;
#pragma unroll
            for (int k = 0; k < kChunkN / 16; ++k) {
                if (16 * k >= Np) break;
                const f4 b = *(const f4 *)(rb + 16 * k);
#pragma unroll
                for (int e = 0; e < 4; ++e) d = __builtin_amdgcn_mfma_f32_16x16x4f32(b[e], ct[k][e], d, 0, 0, 0);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int s = 16 * q + 4 * kg + i;
                m[q][i] = s <= t0 + r16 ? d[i] * expf((float)(lt - steps.l[s])) * steps.dt[s] : 0.0f;
            }
        }
    }
    __syncthreads();
    if constexpr (VEC) {
#pragma unroll
        for (int i = 0; i < NS; ++i) {
            const int n = (threadIdx.x >> 4) + 16 * i, p = 4 * (threadIdx.x & 15);
            if (n < Np) *(f4 *)(sS + n * kLdX + p) = n < N && p < x_width ? rS[i] : (f4){0, 0, 0, 0};
        }
    } else {
        for (int i = threadIdx.x; i < Np * kChunkP; i += 256) {
            const int n = i / kChunkP, p = i % kChunkP;
            sS[n * kLdX + p] = n < N && p < x_width ? st[(size_t)n * P + p] : 0.0f;
        }
    }
    __syncthreads();
    f4 y[kChunkP / 16];
#pragma unroll
    for (int c = 0; c < kChunkP / 16; ++c) y[c] = (f4){0, 0, 0, 0};
#pragma unroll
    for (int k = 0; k < kChunkN / 16; ++k) {
        if (16 * k >= Np) break;
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int c = 0; c < kChunkP / 16; ++c)
                y[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(ct[k][e], sS[(16 * k + 4 * kg + e) * kLdX + 16 * c + r16], y[c], 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float f = expf((float)steps.l[t0 + 4 * kg + i]);
#pragma unroll
        for (int c = 0; c < kChunkP / 16; ++c) y[c][i] *= f;
    }
#pragma unroll
    for (int q = 0; q < kChunk / 16; ++q) {
        if (q > w) break;
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int c = 0; c < kChunkP / 16; ++c)
                y[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(m[q][e], sX[(16 * q + 4 * kg + e) * kLdX + 16 * c + r16], y[c], 0, 0, 0);
    }
    const float Dh = j.D[h];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int tk = t0 + 4 * kg + i;
        if (tk >= cnt) break;
#pragma unroll
        for (int c = 0; c < kChunkP / 16; ++c) {
            const int p = 16 * c + r16;
            if (p < x_width) j.y[(size_t)steps.tok[tk] * sh.inner() + x_col + p] = y[c][i] + Dh * sX[tk * kLdX + p];
        }
    }
}

// A run of one or two chunks: one workgroup walks them for 32 columns of one head; wave w owns the chunk's token tile w. Tokens past the
// run's end count as dt = 0, which leaves everything unchanged. VEC: rows can be read four columns at a time, and the next
// chunk's rows are on their way while a chunk is worked on.
template <bool VEC>
__global__ __launch_bounds__(256) void k_mamba_chunks(MambaJob j) {
    extern __shared__ __attribute__((aligned(16))) float sm[];
    const MambaShape sh = j.sh;
    const int N = sh.state, Np = (N + 15) / 16 * 16, P = sh.vdim, C = sh.channels(), LB = Np + 4;
    const int h = blockIdx.x, g = h / (sh.heads / sh.groups), p0 = blockIdx.y * kWalkP;
    const SeqRun run = j.runs.runs[blockIdx.z];
    if (run.n < kChunkLeast) return;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, r16 = lane & 15, kg = lane >> 4;
    float * sB = sm, * sC = sB + kChunk * LB, * sX = sC + kChunk * LB, * sM = sX + kChunk * 36, * sS = sM + kChunk * 68;
    __shared__ double s_l[kChunk];
    __shared__ float s_dt[kChunk], s_w[kChunk];
    __shared__ int s_tok[kChunk];
    const float a = expf(j.A_log[h]), Dh = j.D[h], bias = j.dt_bias[h];
    float * st = j.state + (((size_t)run.slot * sh.heads + h) * N) * P + p0;
    const int n_tiles = Np / 16;
    // the state in registers: wave w holds row tiles w, w + 4, both column tiles
    f4 S[kChunkN / 64][2];
#pragma unroll
    for (int q = 0; q < kChunkN / 64; ++q)
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int n = (w + 4 * q) * 16 + 4 * kg + i, p = c * 16 + r16;
                S[q][c][i] = (n < N && p0 + p < P && !(run.flags & 1)) ? st[(size_t)n * P + p] : 0.0f;
            }
    constexpr int RB = kChunk * kChunkN / 4 / 256, RX = kChunk * kWalkP / 4 / 256;
    f4 nB[VEC ? RB : 1], nC[VEC ? RB : 1], nX[VEC ? RX : 1];
    float n_dt = 0.0f;
    int n_tok = 0;
    auto token = [&](int base, int tk) { return j.runs.tok[run.start + min(base + tk, run.n - 1)]; };
    auto fetch = [&](int base) {                // of the chunk at base into registers; nothing past the run's end is used
        if (w == 0) {
            n_tok = token(base, lane);
            n_dt = j.proj[(size_t)n_tok * j.ld + sh.inner() + C + h];
        }
        if constexpr (VEC) {
            const int n = 4 * (threadIdx.x & 31);
#pragma unroll
            for (int i = 0; i < RB; ++i) {
                const float * row = j.xbc + (size_t)token(base, (threadIdx.x >> 5) + 8 * i) * C + sh.inner() + g * N + min(n, N - 4);
                nB[i] = *(const f4 *)row;
                nC[i] = *(const f4 *)(row + (size_t)sh.groups * N);
            }
            const int p = 4 * (threadIdx.x & 7);
#pragma unroll
            for (int i = 0; i < RX; ++i)
                nX[i] = *(const f4 *)(j.xbc + (size_t)token(base, (threadIdx.x >> 3) + 32 * i) * C + h * P + min(p0 + p, P - 4));
        }
    };
    fetch(0);
    for (int base = 0; base < run.n; base += kChunk) {
        const int cnt = min(kChunk, run.n - base);
        __syncthreads();
        if (w == 0) {
            s_tok[lane] = n_tok;
            const float dt = lane < cnt ? softplus_f(n_dt + bias) : 0.0f;
            double l = -(double)a * (double)dt;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const double up = __shfl_up(l, o, 64);
                if (lane >= o) l += up;
            }
            s_l[lane] = l;
            s_dt[lane] = dt;
            s_w[lane] = expf((float)(__shfl(l, 63, 64) - l)) * dt;
        }
#pragma unroll
        for (int q = 0; q < kChunkN / 64; ++q)
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int n = (w + 4 * q) * 16 + 4 * kg + i;
                    if (n < Np) sS[n * 36 + c * 16 + r16] = S[q][c][i];
                }
        if constexpr (VEC) {
            const f4 zero = {0, 0, 0, 0};
            const int n = 4 * (threadIdx.x & 31), p = 4 * (threadIdx.x & 7);
            if (n < Np) {
#pragma unroll
                for (int i = 0; i < RB; ++i) {
                    const int tk = (threadIdx.x >> 5) + 8 * i;
                    const bool in = n < N && tk < cnt;
                    *(f4 *)(sB + tk * LB + n) = in ? nB[i] : zero;
                    *(f4 *)(sC + tk * LB + n) = in ? nC[i] : zero;
                }
            }
#pragma unroll
            for (int i = 0; i < RX; ++i) {
                const int tk = (threadIdx.x >> 3) + 32 * i;
                *(f4 *)(sX + tk * 36 + p) = p0 + p < P && tk < cnt ? nX[i] : zero;
            }
        } else {
            __syncthreads();
            for (int i = threadIdx.x; i < kChunk * Np; i += 256) {
                const int tk = i / Np, n = i - tk * Np;
                const float * row = j.xbc + (size_t)s_tok[tk] * C + sh.inner() + g * N + n;
                const bool in = n < N && tk < cnt;
                sB[tk * LB + n] = in ? row[0] : 0.0f;
                sC[tk * LB + n] = in ? row[(size_t)sh.groups * N] : 0.0f;
            }
            for (int i = threadIdx.x; i < kChunk * kWalkP; i += 256) {
                const int tk = i / kWalkP, p = i - tk * kWalkP;
                sX[tk * 36 + p] = (p0 + p < P && tk < cnt) ? j.xbc[(size_t)s_tok[tk] * C + h * P + p0 + p] : 0.0f;
            }
        }
        __syncthreads();
        if (base + kChunk < run.n) fetch(base + kChunk);
        const int t0 = 16 * w;
        double lt[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) lt[i] = s_l[t0 + 4 * kg + i];
        // decayed C B^T of this wave's tokens with everything before them
        for (int q = 0; q <= w; ++q) {
            f4 d = {0, 0, 0, 0};
            const float * ca = sC + (t0 + r16) * LB + 4 * kg, * cb = sB + (16 * q + r16) * LB + 4 * kg;
            for (int k = 0; k < Np; k += 16) {
                const f4 x = *(const f4 *)(ca + k), y = *(const f4 *)(cb + k);
#pragma unroll
                for (int e = 0; e < 4; ++e) d = __builtin_amdgcn_mfma_f32_16x16x4f32(x[e], y[e], d, 0, 0, 0);
            }
            const int sk = 16 * q + r16;
            const double ls = s_l[sk];
            const float dt = s_dt[sk];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int t = t0 + 4 * kg + i;
                sM[t * 68 + sk] = sk <= t ? d[i] * expf((float)(lt[i] - ls)) * dt : 0.0f;
            }
        }
        // (a wave reads only the rows of sM that it wrote)
        f4 y[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
        {
            const float * ca = sC + (t0 + r16) * LB + 4 * kg;
            for (int k = 0; k < Np; k += 16) {
                const f4 x = *(const f4 *)(ca + k);
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int c = 0; c < 2; ++c)
                        y[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[e], sS[(k + 4 * kg + e) * 36 + c * 16 + r16], y[c], 0, 0, 0);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float f = expf((float)lt[i]);
                y[0][i] *= f;
                y[1][i] *= f;
            }
            __builtin_amdgcn_wave_barrier();
            const float * ma = sM + (t0 + r16) * 68 + 4 * kg;
            for (int k = 0; k < t0 + 16; k += 16) {
                const f4 x = *(const f4 *)(ma + k);
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int c = 0; c < 2; ++c)
                        y[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[e], sX[(k + 4 * kg + e) * 36 + c * 16 + r16], y[c], 0, 0, 0);
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int tk = t0 + 4 * kg + i;
            if (tk >= cnt) break;
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const int p = c * 16 + r16;
                if (p0 + p < P) j.y[(size_t)s_tok[tk] * sh.inner() + h * P + p0 + p] = y[c][i] + Dh * sX[tk * 36 + p];
            }
        }
        const float decay = expf((float)s_l[kChunk - 1]);
#pragma unroll
        for (int q = 0; q < kChunkN / 64; ++q) {
            if (w + 4 * q >= n_tiles) break;
            f4 d[2] = {S[q][0] * decay, S[q][1] * decay};
            const int n = (w + 4 * q) * 16 + r16;
            for (int k = 0; k < cnt; k += 4) {
                const int sk = k + kg;
                const float bw = sB[sk * LB + n] * s_w[sk];
#pragma unroll
                for (int c = 0; c < 2; ++c) d[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(bw, sX[sk * 36 + c * 16 + r16], d[c], 0, 0, 0);
            }
            S[q][0] = d[0];
            S[q][1] = d[1];
        }
    }
#pragma unroll
    for (int q = 0; q < kChunkN / 64; ++q)
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int n = (w + 4 * q) * 16 + 4 * kg + i, p = c * 16 + r16;
                if (n < N && p0 + p < P) st[(size_t)n * P + p] = S[q][c][i];
            }
}

template <bool VEC> void launch_chunks(hipStream_t s, const MambaJob & j, int T) {
    const MambaShape & sh = j.sh;
    const int Np = (sh.state + 15) / 16 * 16;
    if (j.runs.longest <= kWalkMost) {
        const size_t lds = ((size_t)2 * kChunk * (Np + 4) + kChunk * 36 + kChunk * 68 + (size_t)Np * 36) * 4;
        constexpr int most = (2 * kChunk * (kChunkN + 4) + kChunk * 36 + kChunk * 68 + kChunkN * 36) * 4;
        static const bool allowed = hipFuncSetAttribute((const void *)k_mamba_chunks<VEC>, hipFuncAttributeMaxDynamicSharedMemorySize, most) == hipSuccess;
        if (!allowed) throw std::runtime_error("mamba2: a chunk does not fit the LDS");
        const dim3 grid((unsigned)sh.heads, (unsigned)((sh.vdim + kWalkP - 1) / kWalkP), (unsigned)j.runs.n);
        hipLaunchKernelGGL(k_mamba_chunks<VEC>, grid, dim3(256), lds, s, j);
        check_launch("mamba_chunks");
        return;
    }
    const dim3 grid((unsigned)sh.heads, (unsigned)((sh.vdim + kChunkP - 1) / kChunkP), (unsigned)(T / kChunk + j.runs.n));
    const size_t lds = (size_t)(kChunk * (Np + 4) + kChunk * kLdX) * 4;
    const size_t lds_out = (size_t)(std::max(kChunk * (Np + 4), Np * kLdX) + kChunk * kLdX) * 4;
    hipLaunchKernelGGL(k_mamba_chunk_sums<VEC>, grid, dim3(256), lds, s, j);
    check_launch("mamba_chunk_sums");
    const unsigned parts = (unsigned)((sh.state * sh.vdim + (VEC ? 1024 : 256) - 1) / (VEC ? 1024 : 256));
    hipLaunchKernelGGL(k_mamba_chunk_states<VEC>, dim3(parts, (unsigned)sh.heads, (unsigned)j.runs.n), dim3(256), 0, s, j);
    check_launch("mamba_chunk_states");
    hipLaunchKernelGGL(k_mamba_chunk_out<VEC>, grid, dim3(256), lds_out, s, j);
    check_launch("mamba_chunk_out");
}

// act[t] = norm over each of the equal parts of (y * silu(z)), times the weight, for parts of up to 1024 columns, a multiple of
// eight: a wave per token and part, which stays in registers. (A workgroup of four waves had two columns per lane to wait for:
// 3321 tokens of eight parts of 512 52 us, a wave
// each 44, with four tokens per workgroup, whose activations are neighbours, 39; a copy of the bytes would take 28.)
template <int ARITH>
__global__ __launch_bounds__(256) void k_mamba_gate_norm_wave(MambaJob j, int T) {
    constexpr int GROUPS = 2;             // of eight columns per lane
    const int inner = j.sh.inner(), len = inner / j.sh.norm_groups;
    // (the activations of four tokens lie side by side)
    const int t = blockIdx.x * 4 + (threadIdx.x >> 6), k0 = blockIdx.y * len, lane = threadIdx.x & 63;
    if (t >= T) return;
    const float * y = j.y + (size_t)t * inner + k0, * z = j.proj + (size_t)t * j.ld + k0, * weight = j.norm_w + k0;
    f4 a[GROUPS][2], b[GROUPS][2], wt[GROUPS][2];
#pragma unroll
    for (int g = 0; g < GROUPS; ++g)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int k = min(8 * (lane + 64 * g), len - 8) + 4 * u;
            a[g][u] = *(const f4 *)(y + k);
            b[g][u] = *(const f4 *)(z + k);
            wt[g][u] = *(const f4 *)(weight + k);
        }
    float q = 0.0f;
#pragma unroll
    for (int g = 0; g < GROUPS; ++g)
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                a[g][u][e] *= silu_f(b[g][u][e]);
                if (8 * (lane + 64 * g) < len) q += a[g][u][e] * a[g][u][e];
            }
    const float inv = 1.0f / sqrtf(wave_sum(q) / (float)len + j.eps);
#pragma unroll
    for (int g = 0; g < GROUPS; ++g) {
        const int k = 8 * (lane + 64 * g);
        if (k >= len) continue;
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = a[g][e / 4][e % 4] * inv * wt[g][e / 4][e % 4];
        store_frag8<ARITH>(j.out, j.out_kf, t, k0 + k, v);
    }
}

// ... and of any other: one workgroup per token and part.
template <int ARITH>
__global__ __launch_bounds__(256) void k_mamba_gate_norm(MambaJob j) {
    extern __shared__ float row[];
    __shared__ float scratch[16];
    const int inner = j.sh.inner(), len = inner / j.sh.norm_groups;
    const int t = blockIdx.x, k0 = blockIdx.y * len;
    const float * y = j.y + (size_t)t * inner + k0, * z = j.proj + (size_t)t * j.ld + k0;
    float q = 0.0f;
    for (int k = threadIdx.x; k < len; k += 256) {
        const float v = y[k] * silu_f(z[k]);
        row[k] = v;
        q += v * v;
    }
    q = block_sum(q, scratch);
    const float inv = 1.0f / sqrtf(q / (float)len + j.eps);
    if (len % 8 == 0 && k0 % 8 == 0) {
        for (int k = 8 * threadIdx.x; k < len; k += 8 * 256) {
            float v[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = row[k + i] * inv * j.norm_w[k0 + k + i];
            store_frag8<ARITH>(j.out, j.out_kf, t, k0 + k, v);
        }
    } else {
        for (int k = threadIdx.x; k < len; k += 256) {
            const float v = row[k] * inv * j.norm_w[k0 + k];
            const size_t at = frag_at(t, k0 + k, j.out_kf);
            if constexpr (ARITH == ARITH_16) ((uint16_t *)j.out)[at] = bf16_bits(v);
            else ((float *)j.out)[at] = v;
        }
    }
}

}  // namespace

size_t mamba_chunk_floats(const MambaShape & sh, int T) {
    return sh.state <= kChunkN ? (size_t)(T / kChunkLeast) * sh.heads * ((size_t)sh.state * sh.vdim + 1) : 0;
}

void mamba_mix(hipStream_t s, int arith, const MambaJob & j, int T) {
    if (j.runs.n <= 0 || T <= 0) return;
    const MambaShape & sh = j.sh;
    if (sh.state > 512) throw std::runtime_error("mamba2: at most 512 state rows per head");
    ShortConv conv;
    conv.runs = j.runs;
    conv.channels = sh.channels(); conv.taps = sh.taps;
    conv.in = j.proj + sh.inner(); conv.ld = j.ld;
    conv.w = j.conv_w; conv.b = j.conv_b;
    conv.state = j.conv_state; conv.plane = j.conv_plane;
    conv.out = j.xbc;
    short_conv(s, conv);
    // Each run by its own length: a decoding row beside prompts takes the walk it takes in a step of its own.
    const bool chunks = j.runs.longest >= kChunkLeast && sh.state <= kChunkN;
    if (!chunks || j.runs.shortest < kChunkLeast) {
        const int below = chunks ? kChunkLeast : INT32_MAX;
        const dim3 grid((unsigned)sh.heads, (unsigned)((sh.vdim + kScanP - 1) / kScanP), (unsigned)j.runs.n);
        const size_t lds = (size_t)(2 * kScanTokens * sh.state + kScanTokens * 256) * 4;
        const int npt = (sh.state + 3) / 4;
        if (npt <= 8) hipLaunchKernelGGL(k_mamba_scan<8>, grid, dim3(256), lds, s, j, below);
        else if (npt <= 16) hipLaunchKernelGGL(k_mamba_scan<16>, grid, dim3(256), lds, s, j, below);
        else if (npt <= 32) hipLaunchKernelGGL(k_mamba_scan<32>, grid, dim3(256), lds, s, j, below);
        else if (npt <= 64) hipLaunchKernelGGL(k_mamba_scan<64>, grid, dim3(256), lds, s, j, below);
        else hipLaunchKernelGGL(k_mamba_scan<128>, grid, dim3(256), lds, s, j, below);
        check_launch("mamba_scan");
    }
    if (chunks) {
        MambaJob c = j;
        c.chunk_decay = c.chunks + (size_t)(T / kChunkLeast) * sh.heads * sh.state * sh.vdim;
        // every row starts at a multiple of four floats
        if (sh.vdim % 4 == 0 && sh.state % 4 == 0) launch_chunks<true>(s, c, T);
        else launch_chunks<false>(s, c, T);
    }
    const int len = sh.inner() / sh.norm_groups;
    if (len % 8 == 0 && len <= 1024 && sh.inner() % 4 == 0 && j.ld % 4 == 0) {
        const dim3 grid((unsigned)((T + 3) / 4), (unsigned)sh.norm_groups);
        if (arith == ARITH_16) hipLaunchKernelGGL(k_mamba_gate_norm_wave<ARITH_16>, grid, dim3(256), 0, s, j, T);
        else hipLaunchKernelGGL(k_mamba_gate_norm_wave<ARITH_32>, grid, dim3(256), 0, s, j, T);
        check_launch("mamba_gate_norm");
        return;
    }
    const dim3 gn((unsigned)T, (unsigned)sh.norm_groups);
    const size_t nl = (size_t)(sh.inner() / sh.norm_groups) * 4;
    if (arith == ARITH_16) hipLaunchKernelGGL(k_mamba_gate_norm<ARITH_16>, gn, dim3(256), nl, s, j);
    else hipLaunchKernelGGL(k_mamba_gate_norm<ARITH_32>, gn, dim3(256), nl, s, j);
    check_launch("mamba_gate_norm");
}

}  // namespace rk

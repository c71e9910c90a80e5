/*
 * Region generation of one integral by one workgroup (gfx950): root, refinement, exact
 * selection of the N - 1 split nodes and the canonical order of the N regions, in one
 * kernel with no other workgroup to wait for.
 *
 * The round kernels (pipeline.h) need two launches per refinement round, and a tree of a
 * few thousand regions is about twenty rounds deep: at that size the launches, their gaps
 * and each round's chain of memory latencies, not the evaluations, are the time.  Here a
 * step costs six barriers of one block:
 *   - every unsplit node that may still be split waits in a pool in LDS (b, slot, dim);
 *   - a histogram in LDS counts all known nodes and the pool by the top bits of b, so one
 *     scan gives theta (a lower bound of the (N-1)-th largest b among the known nodes: what
 *     lies below is dropped) and tau (the M-th largest b of the pool: what lies at or above
 *     is split in this step);
 *   - the step's new nodes are evaluated by every lane, whichever child they are of, and
 *     each child is scored by one lane, all in its registers.
 * What bounds it is the issue rate of one CU: a step of 256 splits at D = 2 (3 blobs, FP32)
 * takes 6.5 us, of it thresholds and pool 1.7, gathering parents 1.2, evaluations 1.4,
 * scores and stores 2.0; the selection and order of 4096 regions 42 us.  Scoring by teams of
 * 8 lanes with the values in LDS (as the round kernels do) took 15 us a step, 3 of 8 lanes
 * idle; one wave's lanes evaluating their own child's nodes was slower for dear integrands.
 * The largest b are split first, M at a time, so few nodes beyond the 2N - 1 that the
 * result needs are made.  The set of regions is the one the rounds give, for any M: see
 * kernels.h for why any order of expansion selects the same N - 1 nodes.
 *
 * A job whose pool reaches Job::grow_stop hands over: its nodes so far become the first
 * candidates of the round kernels.  One that is meant to end here and cannot (pool or tree
 * full, a split too deep) says so, and the rounds generate its batch from the start.
 */
#ifndef VMX_GROW_H
#define VMX_GROW_H

namespace vmx {

constexpr int GROW_WAVES = 8, GROW_THREADS = 64 * GROW_WAVES;
constexpr int GROW_BUCKETS = 4096;
constexpr uint32_t GROW_MAX_NODES = 65535;  // node indexes within a job are 16 bits here
constexpr uint32_t GROW_MAX_REGIONS = 8192;
constexpr uint32_t GROW_DIRECT = 256;  // boundary buckets up to this are ranked directly

/* Buckets of the priorities, 32 per octave over 128 octaves up to `top`; values above
   share the last bucket, values below the first.  lower(k) is at most every value of
   bucket k.  top: the root's b, the largest of a job; 2^32 with the learned priority,
   whose root is infinite and whose size floor (above 2^60) is split first in any order. */
template <typename T>
struct GrowKeys {
    static constexpr int SHIFT = sizeof(T) == 4 ? 18 : 15;  // of the high word: 5 mantissa bits are left
    uint32_t off;
    __device__ static uint32_t high(T b) {
        if constexpr (sizeof(T) == 4)
            return __float_as_uint(float(b));
        else
            return uint32_t(uint64_t(__double_as_longlong(double(b))) >> 32);
    }
    __device__ explicit GrowKeys(T top) {
        const uint32_t k = high(top) >> SHIFT;
        off = k >= uint32_t(GROW_BUCKETS) ? k - uint32_t(GROW_BUCKETS - 1) : 0u;
    }
    __device__ uint32_t bucket(T b) const {
        uint32_t k = high(b) >> SHIFT;
        k = k > off ? k - off : 0u;
        return k < uint32_t(GROW_BUCKETS) ? k : uint32_t(GROW_BUCKETS - 1);
    }
    __device__ T lower(uint32_t k) const {
        if (k == 0) return T(-INFINITY);
        const uint32_t h = (k + off) << SHIFT;
        if constexpr (sizeof(T) == 4)
            return T(__uint_as_float(h));
        else
            return T(__longlong_as_double((long long)(uint64_t(h) << 32)));
    }
};
/* Where bucket k is counted: thread t of the scan holds a run of consecutive buckets, and
   the threads' entries of one place lie side by side, free of bank conflicts. */
__device__ inline uint32_t grow_place(uint32_t k) {
    constexpr uint32_t PER = GROW_BUCKETS / GROW_THREADS;
    return (k % PER) * uint32_t(GROW_THREADS) + (uint32_t(GROW_THREADS) - 1u - k / PER);
}

template <typename T, int D, bool LEARN>
struct GrowShape {
    static constexpr int WAVES = GROW_WAVES, THREADS = GROW_THREADS;
    // FP64 trees of 3 dims: the children's values leave less room for the pool
    static constexpr int POOL = sizeof(T) == 8 && D == 3 ? 1536 : 4096;
    static constexpr int SPLITS = THREADS / 2;  // splits of one step: a lane per child
    static_assert(GROW_BUCKETS % THREADS == 0 && POOL % THREADS == 0, "whole runs per thread");
};

/* The waves' forward passes: a wave takes its lanes' 64 children as four 16-row MFMA
   tiles; the features, then each layer's activations, share one buffer (a layer's operand
   is in registers before its output is written). */
template <int D, int WAVES>
struct GrowNet {
    static constexpr int KP = nn::Dims<D>::KP;
    static_assert(KP + 8 <= nn::WS, "features and activations share rows");
    nn::NetW<KP> net;
    alignas(16) uint16_t act[WAVES][64 * nn::WS];
};

template <typename T, int D, bool LEARN>
struct GrowLds {
    using S = GrowShape<T, D, LEARN>;
    struct Gen {
        uint32_t hist[GROW_BUCKETS];  // low half: known nodes, high half: the pool
        T pool_b[S::POOL];
        uint32_t pool_s[S::POOL];  // node | split dim << 16
        uint32_t list[2 * S::SPLITS];
        T box[S::SPLITS][2 * D];   // of the nodes split in a step: lo, hi
        // the node values of a step's children, as they go to memory; with the learned
        // priority a wave's 64 children use its part of net.act
        T values[LEARN ? 1 : S::WAVES][LEARN ? 1 : 64 * pow3(D)];
        typename std::conditional<LEARN, GrowNet<D, S::WAVES>, char>::type net;
    };
    struct Sel {
        uint64_t split[(GROW_MAX_NODES + 64) / 64];  // bit per node
        uint16_t idx[2][GROW_MAX_REGIONS];           // ping-pong of the sort; idx[1] first lists the bucket
        uint8_t state[GROW_MAX_REGIONS];             // of the bucket's nodes: 0 undecided, 1 split, 2 kept
        T b[GROW_DIRECT];                            // their b, for a direct ranking
        uint32_t key[GROW_MAX_REGIONS];              // the sort's packed codes, and their nodes; codes of ties
        uint16_t node[GROW_MAX_REGIONS];
        uint32_t whist[S::WAVES][256];
        uint32_t digit[256];
        // the second keys of the bucket's nodes, before the sort's lists take the memory
        __device__ T* tie_b1() { return reinterpret_cast<T*>(&idx[0][0]); }
    };
    static_assert(GROW_DIRECT <= GROW_THREADS, "a thread per node of the bucket");
    static_assert(sizeof(uint16_t) * GROW_MAX_REGIONS >= sizeof(T) * GROW_DIRECT && GROW_MAX_REGIONS >= 3 * GROW_DIRECT,
                  "second keys and codes of a bucket");
    union {
        Gen g;
        Sel s;
    };
    __device__ T* child_values(uint32_t ci) {  // of child ci of the step
        if constexpr (LEARN)
            return reinterpret_cast<T*>(&g.net.act[ci / 64][0]) + (ci % 64) * uint32_t(pow3(D));
        else
            return &g.values[ci / 64][(ci % 64) * uint32_t(pow3(D))];
    }
    uint32_t wtot[S::WAVES];
    uint32_t npool[2], nnew[2], nlist[2];  // pool entries kept, children added, splits of a step
    uint32_t kb, above, kt;  // theta's bucket and the nodes above it, tau's bucket
    uint32_t depth[VMX_MAX_DIM];
    uint32_t top_row, nsel, ties, dsel, dabove, dleft, flags;
    uint32_t kor, kand;
    int32_t last;
};

/* A wave's 64 rows of features (`act`, rows of nn::WS) through the network; lane l gets
   row l's raw output.  tiles: 16-row tiles that hold rows in use (uniform).  The operands
   and their order are those of nn::forward_rows; the weights are the first operand, so a
   lane's four results are four neighbouring features of its row, one 8-byte store. */
template <int KP>
__device__ inline float forward_wave(const nn::NetW<KP>& n, uint16_t* act, int tiles, int lane) {
    using nn::bf16x8_t;
    using nn::f32x4_t;
    const int r = lane & 15, kq = (lane >> 4) * 8;
    auto layer = [&](auto ktag, const uint16_t* wt, int ldw, const float* bias) {
        constexpr int K = decltype(ktag)::value;
        bf16x8_t x[4][K / 32];
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int k = 0; k < K / 32; ++k) x[q][k] = nn::ld8(act + (q * 16 + r) * nn::WS + 32 * k + kq);
        team_sync<64>();
#pragma unroll
        for (int ct = 0; ct < nn::W / 16; ++ct) {
            bf16x8_t w[K / 32];
#pragma unroll
            for (int k = 0; k < K / 32; ++k) w[k] = nn::ld8(wt + (ct * 16 + r) * ldw + 32 * k + kq);
            const int f0 = ct * 16 + (lane >> 4) * 4;
            const f32x4_t bv = *reinterpret_cast<const f32x4_t*>(bias + f0);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if (q >= tiles) break;
                f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int k = 0; k < K / 32; ++k)
                    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[k], x[q][k], acc, 0, 0, 0);
                nn::bf16x4_t h;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float z = acc[i] + bv[i];
                    h[i] = __bf16(z > 0.f ? z : 0.f);  // round to nearest even, as nn::f2bf
                }
                *reinterpret_cast<nn::bf16x4_t*>(act + (q * 16 + r) * nn::WS + f0) = h;
            }
        }
        team_sync<64>();
    };
    layer(std::integral_constant<int, KP>{}, &n.w0t[0][0], KP + 8, n.b0);
    layer(std::integral_constant<int, nn::W>{}, &n.w1t[0][0], nn::WS, n.b1);
    layer(std::integral_constant<int, nn::W>{}, &n.w2t[0][0], nn::WS, n.b2);
    float s[4];
#pragma unroll
    for (int part = 0; part < 4; ++part) {
        s[part] = 0.f;
#pragma unroll
        for (int k = 0; k < 16; k += 8) {
            const nn::u16x8_t h =
                *reinterpret_cast<const nn::u16x8_t*>(act + lane * nn::WS + part * 16 + k);
#pragma unroll
            for (int i = 0; i < 8; ++i) s[part] += nn::bf2f(h[i]) * n.w3[part * 16 + k + i];
        }
    }
    team_sync<64>();
    return ((s[0] + s[1]) + (s[2] + s[3])) + n.b3;
}

/* One child of a split, by one lane, all in registers.  The values are held in the frame
   of the split: w[a][j] with a along the split dim and j over the other dims, the lowest
   fastest, so that every index is a constant whatever the dim; only addresses, the
   coordinates and the order of the folds depend on it. */
template <typename T, int D>
struct Child {
    static constexpr int K = pow3(D), KM = pow3(D - 1);
    T w[3][KM];
    T lo[D], hi[D];
    T E[D];                 // folded error along each dim
    float diff[D][KM];      // learned: |Simpson - trapezoid| of the lines along each dim

    int dim;  // the split dim
    __device__ static int other(int i, int dim) { return i < dim ? i : i + 1; }
    /* node index of (a, j) */
    __device__ static int at(int a, int j, int dim) {
        int o = a;
#pragma unroll
        for (int d = 1; d < D; ++d)
            if (dim == d) o = a * pow3(d);
#pragma unroll
        for (int i = 0; i < D - 1; ++i) {
            const int dg = (j / pow3(i)) % 3;
            o += dg * (i < dim ? pow3(i) : pow3(i + 1));
        }
        return o;
    }
    /* a value per dim from one of the split dim and one per other dim */
    template <typename X>
    __device__ static X pick(int d, int dim, X split, const X* others) {
        X r = split;
        if (d < dim) r = others[d < D - 1 ? d : 0];
        if (d > dim) r = others[d > 0 ? d - 1 : 0];
        return r;
    }

    /* child c of the parent with box [plo, phi], split along `split` */
    __device__ void box(const T* plo, const T* phi, int split, int c) {
        dim = split;
#pragma unroll
        for (int d = 0; d < D; ++d) {  // split_boxes
            const T dd = (phi[d] - plo[d]) / T(2);
            const T mid = plo[d] + dd * T(1);
            lo[d] = d == dim && c == 1 ? mid : plo[d];
            hi[d] = d == dim && c == 0 ? mid : phi[d];
        }
    }
    __device__ void read(const T* v) {
#pragma unroll
        for (int a = 0; a < 3; ++a)
#pragma unroll
            for (int j = 0; j < KM; ++j) w[a][j] = v[at(a, j, dim)];
    }

    __device__ static T line(T p0, T p1, T p2, int heur, float& d) {
        const T sm = simpson(p0, p1, p2), tz = trapezoid(p0, p2);
        d = vabs(float(sm) - float(tz));
        return heur == 0 ? metric_relative(sm, tz) : metric_absolute(sm, tz);
    }

    /* heuristic error and split dim; also fills E and, for the learned priority, diff */
    __device__ void score(int heur, T& e, int& dm) {
        T Es, Eo[D > 1 ? D - 1 : 1];
        float ds[KM], dq[D > 1 ? D - 1 : 1][KM];
        Eo[0] = T(0);
        {
            T m[KM];
#pragma unroll
            for (int j = 0; j < KM; ++j) m[j] = line(w[0][j], w[1][j], w[2][j], heur, ds[j]);
#pragma unroll
            for (int n = KM / 3; n >= 1; n /= 3)
#pragma unroll
                for (int q = 0; q < n; ++q) m[q] = simpson(m[3 * q], m[3 * q + 1], m[3 * q + 2]);
            Es = m[0];
        }
        if constexpr (D == 2) {
            T m[3];
#pragma unroll
            for (int a = 0; a < 3; ++a) m[a] = line(w[a][0], w[a][1], w[a][2], heur, dq[0][a]);
            Eo[0] = simpson(m[0], m[1], m[2]);
        } else if constexpr (D == 3) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                // lines along other dim i; what remains is the split dim (a) and the other
                // other dim (b), folded lower dim first
                const bool split_first = dim < other(1 - i, dim);
                T m[3][3];
                float un;
#pragma unroll
                for (int a = 0; a < 3; ++a)
#pragma unroll
                    for (int b = 0; b < 3; ++b) {
                        const int j0 = i == 0 ? 3 * b : b, sj = i == 0 ? 1 : 3;
                        m[a][b] = line(w[a][j0], w[a][j0 + sj], w[a][j0 + 2 * sj], heur, un);
                    }
                T r[3];
#pragma unroll
                for (int y = 0; y < 3; ++y) {
                    const T n0 = split_first ? m[0][y] : m[y][0], n1 = split_first ? m[1][y] : m[y][1],
                            n2 = split_first ? m[2][y] : m[y][2];
                    r[y] = simpson(n0, n1, n2);
                }
                Eo[i] = simpson(r[0], r[1], r[2]);
            }
        }
#pragma unroll
        for (int d = 0; d < D; ++d) {
            E[d] = pick(d, dim, Es, Eo);
#pragma unroll
            for (int j = 0; j < KM; ++j) {
                if constexpr (D == 2)
                    diff[d][j] = d == dim ? ds[j] : dq[0][j];
                else
                    diff[d][j] = ds[j];  // learned priority: D <= 2
            }
        }
        heuristic_pick<T, D>(E, 1, lo, hi, heur, e, dm);
    }

    /* nn::region_features as BF16 into row; gives its s and total depth */
    __device__ void features(const Job<T>& jb, const uint32_t* pcode, uint16_t* row, float& s, int& depth) const {
        constexpr int KP = nn::Dims<D>::KP;
        s = 0.f;
#pragma unroll
        for (int a = 0; a < 3; ++a)
#pragma unroll
            for (int j = 0; j < KM; ++j) s = vmax(s, vabs(float(w[a][j])));
        const float inv = 1.f / vmax(s, 0x1p-100f);
        depth = 0;
#pragma unroll
        for (int d = 0; d < D; ++d) {
            const T c = T((T(0.5) * (lo[d] + hi[d]) - jb.lo[d]) / (jb.hi[d] - jb.lo[d]));
            const int n = nn::code_depth(pcode[d]) + (d == dim ? 1 : 0);
            depth += n;
            row[d] = nn::f2bf(float(c));
            row[D + d] = nn::f2bf(-float(n) * (1.f / 16.f));
            row[2 * D + d] = nn::f2bf((jb.lres[d] - float(n)) * (1.f / 16.f));
            float acc = 0.f;
#pragma unroll
            for (int jl = 0; jl < KM; ++jl) {
                float wt = 1.f;
#pragma unroll
                for (int e = 0; e < D - 1; ++e) wt *= (jl / pow3(e)) % 3 == 1 ? (4.f / 6.f) : (1.f / 6.f);
                acc += wt * diff[d][jl];
            }
            row[3 * D + K + d] = nn::f2bf(acc * inv);
        }
#pragma unroll
        for (int a = 0; a < 3; ++a)
#pragma unroll
            for (int j = 0; j < KM; ++j) row[3 * D + at(a, j, dim)] = nn::f2bf(float(w[a][j]) * inv);
        row[4 * D + K] = nn::f2bf(float(depth) * (1.f / 32.f));
        static_assert((4 * D + K + 1) % 2 == 0, "the padding starts at a 4-byte boundary");
#pragma unroll
        for (int i = 4 * D + K + 1; i < KP; i += 2) *reinterpret_cast<uint32_t*>(row + i) = 0;
    }
};

/* Inclusive sum over the lanes of a wave below and at this one, and over 16 lanes. */
template <int CTRL, int ROWS>
__device__ inline uint32_t dpp_add(uint32_t v) {
    return v + uint32_t(__builtin_amdgcn_update_dpp(0, int(v), CTRL, ROWS, 0xF, false));
}
__device__ inline uint32_t row_scan(uint32_t v) {
    v = dpp_add<0x111, 0xF>(v);  // row_shr:1, :2, :4, :8
    v = dpp_add<0x112, 0xF>(v);
    v = dpp_add<0x114, 0xF>(v);
    return dpp_add<0x118, 0xF>(v);
}
__device__ inline uint32_t wave_scan(uint32_t v) {
    v = row_scan(v);
    v = dpp_add<0x142, 0xA>(v);     // row_bcast:15 into rows 1 and 3
    return dpp_add<0x143, 0xC>(v);  // row_bcast:31 into rows 2 and 3
}

/* A barrier of the block that orders LDS only: global stores stay in flight across it. */
__device__ inline void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

/* theta and tau from the histogram: kb = the bucket of the need-th largest b of all known
   nodes (NONE if fewer are known) with `above` nodes in higher buckets, kt = the bucket of
   the want-th largest b of the pool (0 if the pool is smaller).  Two barriers. */
template <typename T, int D, bool LEARN>
__device__ inline void grow_thresholds(GrowLds<T, D, LEARN>& L, uint32_t need, uint32_t want) {
    using S = GrowShape<T, D, LEARN>;
    constexpr int PER = GROW_BUCKETS / S::THREADS;
    static_assert(S::WAVES <= 16, "the waves' totals are scanned in one row of lanes");
    const int t = int(threadIdx.x), lane = t & 63, wave = t >> 6;
    const int first = (S::THREADS - 1 - t) * PER;  // thread 0 holds the highest buckets
    uint32_t v[PER], sum = 0;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        v[i] = L.g.hist[i * S::THREADS + t];
        sum += v[i];
    }
    const uint32_t incl = wave_scan(sum);  // both halves at once: neither total passes 16 bits
    if (lane == 63) L.wtot[wave] = incl;
    if (t == 0) {
        L.kb = NONE;
        L.above = 0;
        L.kt = 0;
    }
    lds_barrier();
    const uint32_t tot = row_scan(lane < S::WAVES ? L.wtot[lane] : 0u);
    uint32_t hi = incl - sum;  // of the buckets above this thread's
    if (wave > 0) hi += uint32_t(__builtin_amdgcn_readlane(int(tot), __builtin_amdgcn_readfirstlane(wave) - 1));
    const uint32_t a0 = hi & 0xFFFFu, a1 = a0 + (sum & 0xFFFFu), p0 = hi >> 16, p1 = p0 + (sum >> 16);
    if (a0 < need && need <= a1) {
        uint32_t acc = a0;
#pragma unroll
        for (int i = PER - 1; i >= 0; --i) {
            const uint32_t c = v[i] & 0xFFFFu;
            if (acc < need && need <= acc + c) {
                L.kb = uint32_t(first + i);
                L.above = acc;
            }
            acc += c;
        }
    }
    if (p0 < want && want <= p1) {
        uint32_t acc = p0;
#pragma unroll
        for (int i = PER - 1; i >= 0; --i) {
            const uint32_t c = v[i] >> 16;
            if (acc < want && want <= acc + c) L.kt = uint32_t(first + i);
            acc += c;
        }
    }
    lds_barrier();
}

/* Word w of the full key (b, b1, ~codes) of the node in slot s, the most significant first. */
template <typename T, int D>
__device__ inline uint32_t grow_key_word(const TreeArrays<T>& t, size_t s, int w) {
    constexpr int W = int(sizeof(T)) / 4;
    if (w >= 2 * W) return ~t.code[s * D + (w - 2 * W)];
    const T v = w < W ? t.b[s] : t.b1[s];
    if constexpr (W == 1)
        return __float_as_uint(float(v));
    else
        return uint32_t(uint64_t(__double_as_longlong(double(v))) >> (w % W == 0 ? 32 : 0));
}

/* Exact selection and canonical order of a job that has grown to the end: the nodes above
   theta's bucket are split, the (need - above) largest of it too by the full key
   (b, b1, ~codes), and the unsplit children of split nodes, sorted by (code_0, ...,
   code_{D-1}), are the regions.  Returns the number of regions (uniform). */
template <typename T, int D, bool LEARN>
__device__ inline uint32_t grow_select(GrowLds<T, D, LEARN>& L, const TreeArrays<T>& t, const GrowKeys<T>& keys,
                                       uint32_t base, uint32_t count, uint32_t need, int32_t* __restrict__ leaf) {
    using S = GrowShape<T, D, LEARN>;
    constexpr int NT = S::THREADS;
    const int tid = int(threadIdx.x), lane = tid & 63, wave = tid >> 6;
    const uint32_t kb = L.kb, above = L.above;
    const uint32_t whole = (count + uint32_t(NT) - 1) / uint32_t(NT) * uint32_t(NT);  // whole waves
    __syncthreads();  // the pool's memory becomes the selection's
    constexpr int AHEAD = 8;  // loads in flight: the passes over the nodes are else all latency
    for (uint32_t i0 = tid; i0 < whole; i0 += AHEAD * NT) {
        T b[AHEAD];
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
            const uint32_t i = i0 + uint32_t(u * NT);
            b[u] = i < count ? t.b[base + i] : T(0);
        }
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
            const uint32_t i = i0 + uint32_t(u * NT);
            if (i >= whole) break;  // whole waves
            const uint32_t k = keys.bucket(b[u]);
            const bool have = i < count && need > 0, in = have && k == kb;
            const uint64_t m = __ballot(have && k > kb);
            if (lane == 0) L.s.split[i >> 6] = m;
            const uint32_t pos = wave_append(in, &L.nsel);
            if (in && pos < GROW_MAX_REGIONS) {
                L.s.idx[1][pos] = uint16_t(i);
                L.s.state[pos] = 0;
            }
        }
    }
    __syncthreads();
    const uint32_t nb = L.nsel;
    if (nb > GROW_MAX_REGIONS) return NONE;  // uniform: more ties than the list holds
    if (need > 0) {
        const uint32_t take = need - above;  // this many of the bucket's nodes are split
        if (nb <= GROW_DIRECT) {
            // each node's place by counting the larger keys; b decides nearly always, and where
            // some tie (siblings that inherit their parent's b) the rest of their keys come to
            // LDS too
            const uint32_t i = uint32_t(tid);
            const bool own = i < nb;
            const T bi = own ? t.b[base + L.s.idx[1][i]] : T(0);
            if (own) L.s.b[i] = bi;
            __syncthreads();
            uint32_t larger = 0;
            bool tied = false;
            for (uint32_t k = 0; k < nb; ++k) {
                const T bk = L.s.b[k];
                larger += bk > bi ? 1u : 0u;
                tied |= bk == bi && k != i;
            }
            if (__syncthreads_or(own && tied)) {
                T* const b1 = L.s.tie_b1();
                uint32_t* const code = L.s.key;
                T b1i = T(0);
                uint32_t ci[D] = {};
                if (own) {
                    const size_t s = size_t(base) + L.s.idx[1][i];
                    b1[i] = b1i = t.b1[s];
#pragma unroll
                    for (int d = 0; d < D; ++d) code[uint32_t(d) * GROW_DIRECT + i] = ci[d] = t.code[s * D + d];
                }
                __syncthreads();
                for (uint32_t k = 0; k < nb; ++k) {
                    const T b1k = b1[k];
                    bool same = true, first = false;  // smaller codes first
#pragma unroll
                    for (int d = 0; d < D; ++d) {
                        const uint32_t ck = code[uint32_t(d) * GROW_DIRECT + k];
                        first |= same && ck < ci[d];
                        same &= ck == ci[d];
                    }
                    larger += L.s.b[k] == bi && (b1k > b1i || (b1k == b1i && first)) ? 1u : 0u;
                }
            }
            if (own) {
                const uint32_t x = L.s.idx[1][i];
                L.s.state[i] = larger < take ? 1 : 2;
                if (larger + 1 == take) L.last = int32_t(x);
                if (larger < take) atomicOr(reinterpret_cast<unsigned long long*>(&L.s.split[x >> 6]), 1ull << (x & 63));
            }
        } else {
            // radix selection over the keys' 32-bit words, a byte per pass, until one
            // undecided node is left (keys are unique).  A thread's nodes and their current
            // word are in registers, and bytes that all undecided nodes share are passed
            // over: regions of a size over flat parts differ in their codes alone.  The whole
            // kernel, for a constant (1024 tied nodes in the bucket: 2 dims, FP64, 1600 regions,
            // and 3 dims) 727 -> 125 and 1042 -> 338 us, against buckets of up to 1024 ranked
            // directly with the ties' keys in device memory; 2 dims, FP32, 300 regions (768
            // nodes) 476 -> 90; a polynomial of 4000 regions 219 -> 216 (ranking costs the
            // square of the bucket: 55 us at 1024 nodes without ties, a pass here 4)
            constexpr int W = int(sizeof(T)) / 4, PER = int(GROW_MAX_REGIONS) / NT;
            uint32_t x[PER], word[PER], open = 0, up = 0;  // open, up: bit per own node
#pragma unroll
            for (int r = 0; r < PER; ++r) {
                const uint32_t i = uint32_t(r * NT + tid);
                x[r] = i < nb ? uint32_t(L.s.idx[1][i]) : 0u;
                open |= i < nb ? 1u << r : 0u;
            }
            uint32_t rank = take, left = nb;
            for (int w = 0; w < 2 * W + D && left > 1; ++w) {
                if (tid == 0) {
                    L.kor = 0;
                    L.kand = NONE;
                }
                uint32_t any = 0, all = NONE;
#pragma unroll
                for (int r = 0; r < PER; ++r) word[r] = open >> r & 1u ? grow_key_word<T, D>(t, size_t(base) + x[r], w) : 0u;
#pragma unroll
                for (int r = 0; r < PER; ++r)
                    if (open >> r & 1u) {
                        any |= word[r];
                        all &= word[r];
                    }
                for (int o = 32; o > 0; o >>= 1) {
                    any |= uint32_t(__shfl_xor(int(any), o, 64));
                    all &= uint32_t(__shfl_xor(int(all), o, 64));
                }
                __syncthreads();
                if (lane == 0) {
                    atomicOr(&L.kor, any);
                    atomicAnd(&L.kand, all);
                }
                __syncthreads();
                const uint32_t differ = L.kor ^ L.kand;
                for (int sh = differ ? (31 - __clz(int(differ))) & ~7 : -1; sh >= 0 && left > 1; sh -= 8) {
                    if ((differ >> sh & 0xFFu) == 0) continue;
                    if (tid < 256) L.s.digit[tid] = 0;
                    __syncthreads();
#pragma unroll
                    for (int r = 0; r < PER; ++r)
                        if (open >> r & 1u) atomicAdd(&L.s.digit[word[r] >> sh & 0xFFu], 1u);
                    __syncthreads();
                    const uint32_t own = tid < 256 ? L.s.digit[tid] : 0u;
                    __syncthreads();
                    suffix_sum256(L.s.digit);
                    if (tid < 256 && L.s.digit[tid] >= rank && (tid == 255 || L.s.digit[tid + 1] < rank)) {
                        L.dsel = uint32_t(tid);
                        L.dabove = L.s.digit[tid] - own;
                        L.dleft = own;
                    }
                    __syncthreads();
                    const uint32_t dsel = L.dsel;
#pragma unroll
                    for (int r = 0; r < PER; ++r)
                        if (open >> r & 1u) {
                            const uint32_t dg = word[r] >> sh & 0xFFu;
                            if (dg != dsel) open &= ~(1u << r);
                            if (dg > dsel) up |= 1u << r;
                        }
                    rank -= L.dabove;
                    left = L.dleft;
                    __syncthreads();
                }
                __syncthreads();
            }
#pragma unroll
            for (int r = 0; r < PER; ++r) {
                const uint32_t i = uint32_t(r * NT + tid);
                if (i >= nb) break;
                if (open >> r & 1u) L.last = int32_t(x[r]);
                const bool split = (open | up) >> r & 1u;
                L.s.state[i] = split ? 1 : 2;
                if (split) atomicOr(reinterpret_cast<unsigned long long*>(&L.s.split[x[r] >> 6]), 1ull << (x[r] & 63));
            }
        }
        __syncthreads();
        if (L.last >= 0) {
            const T bk = t.b[base + L.last], b1k = t.b1[base + L.last];
            for (uint32_t i = tid; i < nb; i += NT) {
                const size_t s = size_t(base) + L.s.idx[1][i];
                if (L.s.state[i] == 2 && t.b[s] == bk && t.b1[s] == b1k) atomicAdd(&L.ties, 1u);
            }
        }
        __syncthreads();
    }
    if (tid == 0) L.nsel = 0;
    __syncthreads();
    for (uint32_t i0 = tid; i0 < whole; i0 += AHEAD * NT) {
        int32_t parent[AHEAD];
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
            const uint32_t i = i0 + uint32_t(u * NT);
            parent[u] = i < count ? t.parent[base + i] : -1;
        }
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
            const uint32_t i = i0 + uint32_t(u * NT);
            if (i >= whole) break;
            bool is = false;
            if (i < count && !((L.s.split[i >> 6] >> (i & 63)) & 1u)) {
                const uint32_t q = parent[u] >= 0 ? uint32_t(parent[u]) - base : 0u;
                is = parent[u] >= 0 ? (L.s.split[q >> 6] >> (q & 63)) & 1u : need == 0;
            }
            const uint32_t pos = wave_append(is, &L.nsel);
            if (is && pos < GROW_MAX_REGIONS) L.s.idx[0][pos] = uint16_t(i);
        }
    }
    __syncthreads();
    const uint32_t n = L.nsel;
    if (n != need + 1) return n;
    // least significant byte first; each wave ranks a contiguous run of positions, so every
    // pass keeps the order of equal digits.  The key is (code_0, ..., code_{D-1}) in fields
    // as wide as the deepest split where that fits 32 bits, packed in LDS once; else one
    // dim's codes after the other, the last first, from memory.
    constexpr int ROUNDS = int(GROW_MAX_REGIONS) / NT;
    const uint32_t run = (n + uint32_t(NT) - 1) / uint32_t(NT) * 64u;  // positions per wave
    int width = 0;
#pragma unroll
    for (int d = 0; d < D; ++d) width += L.depth[d] ? int(L.depth[d]) + 1 : 0;
    const bool packed = width <= 32;
    if (packed) {
        for (uint32_t p = tid; p < n; p += NT) {
            const size_t s = size_t(base) + L.s.idx[0][p];
            uint32_t key = 0;
#pragma unroll
            for (int d = 0; d < D; ++d)
                if (L.depth[d]) key = uint32_t(uint64_t(key) << (L.depth[d] + 1)) | t.code[s * D + d];
            L.s.key[p] = key;
            L.s.node[p] = L.s.idx[0][p];
        }
        __syncthreads();
    }
    int cur = 0;
    for (int d = packed ? 0 : D - 1; d >= 0; --d) {
        if (!packed && L.depth[d] == 0) continue;  // every code is 1
        const int bits = packed ? width : int(L.depth[d]) + 1;
        for (int sh = 0; sh < bits; sh += 8) {
            for (int i = tid; i < S::WAVES * 256; i += NT) (&L.s.whist[0][0])[i] = 0;
            __syncthreads();
            uint32_t item[ROUNDS], dg[ROUNDS], rk[ROUNDS];
#pragma unroll
            for (int r = 0; r < ROUNDS; ++r) {
                const uint32_t p = uint32_t(wave) * run + uint32_t(r) * 64u + uint32_t(lane);
                const bool ok = uint32_t(r) * 64u < run && p < n;
                // packed: items are places in key[], which starts in the list's order
                item[r] = !ok ? NONE : (packed && sh == 0 ? p : uint32_t(L.s.idx[cur][p]));
                const uint32_t key = !ok ? 0u : (packed ? L.s.key[item[r]] : t.code[(size_t(base) + item[r]) * D + d]);
                dg[r] = (key >> sh) & 0xFFu;
            }
#pragma unroll
            for (int r = 0; r < ROUNDS; ++r) {
                if (uint32_t(r) * 64u >= run) break;  // uniform
                const bool ok = item[r] != NONE;
                uint64_t same = __ballot(ok);
#pragma unroll
                for (int b = 0; b < 8; ++b) {
                    const uint64_t m = __ballot((dg[r] >> b) & 1u);
                    same &= (dg[r] >> b) & 1u ? m : ~m;
                }
                const uint64_t below = same & ((1ull << lane) - 1ull);
                const uint32_t old = L.s.whist[wave][dg[r]];
                rk[r] = old + uint32_t(__popcll(below));
                team_sync<64>();
                if (ok && below == 0) L.s.whist[wave][dg[r]] = old + uint32_t(__popcll(same));
                team_sync<64>();
            }
            __syncthreads();
            // exclusive starts per (digit, wave)
            uint32_t tot = 0;
            if (tid < 256) {
                for (int w = 0; w < S::WAVES; ++w) {
                    const uint32_t c = L.s.whist[w][tid];
                    L.s.whist[w][tid] = tot;
                    tot += c;
                }
            }
            uint32_t incl = tot;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const uint32_t u = __shfl_up(incl, o, 64);
                if (lane >= o) incl += u;
            }
            if (lane == 63 && wave < 4) L.wtot[wave] = incl;
            __syncthreads();
            if (tid < 256) {
                uint32_t start = incl - tot;
                for (int w = 0; w < wave; ++w) start += L.wtot[w];
                L.s.digit[tid] = start;
            }
            __syncthreads();
#pragma unroll
            for (int r = 0; r < ROUNDS; ++r)
                if (item[r] != NONE)
                    L.s.idx[cur ^ 1][L.s.digit[dg[r]] + L.s.whist[wave][dg[r]] + rk[r]] = uint16_t(item[r]);
            __syncthreads();
            cur ^= 1;
        }
    }
    for (uint32_t p = tid; p < n; p += NT)
        leaf[p] = int32_t(base + (packed ? L.s.node[width > 0 ? L.s.idx[cur][p] : p] : L.s.idx[cur][p]));
    return n;
}

/* select = 1: every job is meant to end here, and its regions' slots go to
   leaf[reg_base ..] in canonical order (-1 everywhere, with JF_HANDOVER, if it could not);
   0: growth only, and the job's state is left as the round kernels expect it, with its
   nodes as the first round's candidates unless it grew to the end. */
template <typename T, int D, typename F, typename M, bool LEARN>
__global__ void __launch_bounds__(GROW_THREADS)
    k_grow(GenArgs<T> g, const F* __restrict__ fs, int32_t* __restrict__ leaf, int select) {
    using S = GrowShape<T, D, LEARN>;
    constexpr int K = pow3(D), NT = S::THREADS, PPT = S::POOL / NT;
    __shared__ GrowLds<T, D, LEARN> L;
    const uint32_t j = blockIdx.x;
    const Job<T>& jb = g.jobs[j];
    const F& f = fs[j];
    const TreeArrays<T> t = g.t;
    const uint64_t start = wall_clock64();
    const uint32_t base = jb.node_base, need = jb.N - 1;
    const uint32_t cap = jb.node_cap < GROW_MAX_NODES ? jb.node_cap : GROW_MAX_NODES;
    const int tid = int(threadIdx.x), lane = tid & 63, wave = tid >> 6;

    // ---- root
    for (int i = tid; i < GROW_BUCKETS; i += NT) L.g.hist[i] = 0;
    if (tid < 2) L.npool[tid] = L.nnew[tid] = L.nlist[tid] = 0;
    if (tid < VMX_MAX_DIM) L.depth[tid] = 0;
    if (tid == 0) {
        L.top_row = L.nsel = L.ties = L.flags = 0;
        L.last = -1;
    }
    if constexpr (LEARN) {
        const uint4* src = static_cast<const uint4*>(g.net);
        uint4* dst = reinterpret_cast<uint4*>(&L.g.net.net);
        for (int i = tid; i < int(sizeof(L.g.net.net) / 16); i += NT) dst[i] = src[i];
    }
    T* const rv = reinterpret_cast<T*>(L.g.pool_b);  // the root's values, before the pool's first use
    for (int idx = tid; idx < K; idx += NT) {
        T x[D];
        for (int d = 0; d < D; ++d) x[d] = node_coord<T>(double(digit3(idx, d)) / 2.0, jb.lo[d], jb.hi[d]);
        const T y = f.template eval<Ahead<M>, D>(x);
        rv[idx] = y;
        t.v[size_t(base) * K + idx] = y;
    }
    if (tid < D) {
        t.lo[size_t(base) * D + tid] = jb.lo[tid];
        t.hi[size_t(base) * D + tid] = jb.hi[tid];
        t.code[size_t(base) * D + tid] = 1u;
    }
    __syncthreads();
    if (tid == 0) {
        Child<T, D> ch;
        T e;
        int dm;
        ch.dim = 0;
        ch.read(rv);
#pragma unroll
        for (int d = 0; d < D; ++d) {
            ch.lo[d] = jb.lo[d];
            ch.hi[d] = jb.hi[d];
        }
        ch.score(jb.heur, e, dm);
        // with a learned priority the root goes first whatever its score (k_roots)
        const T pe = jb.learn ? T(INFINITY) : e;
        t.err[base] = pe;
        if (jb.learn && jb.lfloor > 0) dm = 0;
        t.dim[base] = dm;
        t.b[base] = pe;
        t.b1[base] = T(INFINITY);
        t.parent[base] = -1;
        t.child[base] = -1;
        t.job[base] = j;
        L.g.hist[grow_place(GrowKeys<T>(jb.learn ? T(0x1p32) : pe).bucket(pe))] = need > 0 ? 0x10001u : 1u;
        L.g.pool_b[0] = pe;
        if (need > 0) {
            L.g.pool_s[0] = uint32_t(dm) << 16;
            L.npool[0] = 1;
        }
    }
    __syncthreads();

    // ---- growth
    const GrowKeys<T> keys(jb.learn ? T(0x1p32) : L.g.pool_b[0]);
    uint32_t count = 1, steps = 0, deepest[D] = {};
    int par = 0;
    bool done = false;
    const uint32_t stop = jb.grow_stop;
    for (;;) {
        // the pool into registers, while the thresholds are found
        const uint32_t np = L.npool[par] + L.nnew[par];
        T pb[PPT];
        uint32_t ps[PPT];
#pragma unroll
        for (int i = 0; i < PPT; ++i) {
            const uint32_t q = uint32_t(i * NT + tid);
            pb[i] = q < np ? L.g.pool_b[q] : T(0);
            ps[i] = q < np ? L.g.pool_s[q] : NONE;
        }
        // every wave busy until the end is near, then half: fewer splits too many; deepened
        // steps take two passes of splits, whose children wait for the next step
        const bool all = need > (count - 1) / 2 + 2 * uint32_t(S::SPLITS);
        const uint32_t most = uint32_t(S::SPLITS) * (g.deepen ? 2u : 1u);
        grow_thresholds<T, D, LEARN>(L, need, all ? most : most / 2);
        done = np == 0;
        if (done || np >= stop) break;  // uniform
        const T th = L.kb != NONE ? keys.lower(L.kb) : T(-INFINITY), tau = keys.lower(L.kt);
        const T eff = tau > th ? tau : th;
#pragma unroll
        for (int i = 0; i < PPT; ++i) {
            if (uint32_t(i * NT) >= np) break;  // uniform
            const bool have = ps[i] != NONE;
            bool split = have && pb[i] >= eff;
            const uint32_t at = wave_append(split, &L.nlist[par]);
            if (split && at >= most) split = false;  // the rest of tau's bucket waits
            if (split) L.g.list[at] = ps[i];
            const bool keep = have && !split && pb[i] >= th;
            const uint32_t k = wave_append(keep, &L.npool[par ^ 1]);
            if (keep) {
                L.g.pool_b[k] = pb[i];
                L.g.pool_s[k] = ps[i];
            } else if (have) {
                atomicSub(&L.g.hist[grow_place(keys.bucket(pb[i]))], 0x10000u);
            }
        }
        __syncthreads();
        const uint32_t listed = L.nlist[par] < most ? L.nlist[par] : most;
        const uint32_t kept = L.npool[par ^ 1];
        par ^= 1;
        if (tid == 0) {  // the counters the next step fills
            L.nlist[par] = 0;
            L.npool[par ^ 1] = L.nnew[par ^ 1] = 0;
        }
        // room for the children, in the tree and in the pool (uniform)
        if (count + 2 * listed > cap) {
            if (tid == 0) L.flags |= count + 2 * listed > jb.node_cap ? JF_CAPACITY : 0u;
            break;
        }
        if (kept + 2 * listed > uint32_t(S::POOL)) break;
        ++steps;
        for (uint32_t l0 = 0; l0 < listed; l0 += uint32_t(S::SPLITS)) {
            const uint32_t nl = listed - l0 < uint32_t(S::SPLITS) ? listed - l0 : uint32_t(S::SPLITS);
            const uint32_t* list = L.g.list + l0;
            // the children's node values gather in LDS as they go to memory, every lane at work
            // whichever child a node is of: the planes they inherit (consecutive lanes,
            // consecutive nodes), then the new ones (a handful of splits would else evaluate
            // 3^(D-1) nodes one after the other).  A lane per child loads the rest meanwhile.
            constexpr uint32_t KM = uint32_t(pow3(D - 1));
            const uint32_t it = uint32_t(tid) / 2u;
            const int c = tid & 1;
            const bool go = it < nl;
            const uint32_t entry = go ? list[it] : 0u;
            const uint32_t node = base + (entry & 0xFFFFu);
            T plo[D], phi[D], bp = T(0), b1p = T(0), errp = T(0);
            uint32_t pcode[D];
            if (go) {
#pragma unroll
                for (int d = 0; d < D; ++d) {
                    plo[d] = t.lo[size_t(node) * D + d];
                    phi[d] = t.hi[size_t(node) * D + d];
                    pcode[d] = t.code[size_t(node) * D + d];
                }
                bp = t.b[node];
                b1p = t.b1[node];
                if constexpr (LEARN) errp = t.err[node];
            }
            for (uint32_t q0 = uint32_t(tid); q0 < nl * 4u * KM; q0 += 4u * uint32_t(NT)) {
                T val[4];
                T* at[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {  // four loads in flight
                    const uint32_t q = q0 + uint32_t(u * NT);
                    at[u] = nullptr;
                    if (q >= nl * 4u * KM) continue;
                    const uint32_t ci = q / (2u * KM), en = list[ci / 2u];
                    const int j0 = int(q % KM), far = int(q / KM) & 1, dim = int(en >> 16);  // plane 0 or 2 of the child
                    at[u] = L.child_values(ci) + Child<T, D>::at(2 * far, j0, dim);
                    val[u] = t.v[(size_t(base) + (en & 0xFFFFu)) * K + Child<T, D>::at(int(ci & 1u) + far, j0, dim)];
                }
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (at[u]) *at[u] = val[u];
            }
            if (go && c == 0) {
#pragma unroll
                for (int d = 0; d < D; ++d) {
                    L.g.box[it][d] = plo[d];
                    L.g.box[it][D + d] = phi[d];
                }
            }
            lds_barrier();
            for (uint32_t q = uint32_t(tid); q < nl * 2u * KM; q += uint32_t(NT)) {
                const uint32_t ci = q / KM;
                const int dim = int(list[ci / 2u] >> 16);
                T lo[D], hi[D], x[D];
#pragma unroll
                for (int d = 0; d < D; ++d) {
                    lo[d] = L.g.box[ci / 2u][d];
                    hi[d] = L.g.box[ci / 2u][D + d];
                }
                split_new_node<T, D>(lo, hi, dim, int(ci & 1u), int(q % KM), x);
                L.child_values(ci)[Child<T, D>::at(1, int(q % KM), dim)] = f.template eval<Ahead<M>, D>(x);
            }
            lds_barrier();
            if (uint32_t(wave) * 32u < nl) {
                const size_t s = size_t(base) + count + 2 * it + c;
                Child<T, D> ch;
                T e = T(0), nb = T(0), nb1 = T(0);
                int dm = 0, fd = 0;
                float sc = 0.f;
                bool pool = false;
                uint16_t* row = nullptr;
                if constexpr (LEARN) row = &L.g.net.act[wave][lane * nn::WS];
                {
                    const uint32_t c0 = uint32_t(wave) * 64u, nc = 2u * nl - c0 < 64u ? 2u * nl - c0 : 64u;
                    const T* from = L.child_values(c0);
                    T* to = t.v + (size_t(base) + count + c0) * K;
                    for (uint32_t q = uint32_t(lane); q < nc * uint32_t(K); q += 64u) to[q] = from[q];
                }
                if (go) {
                    ch.box(plo, phi, int(entry >> 16), c);
                    ch.read(L.child_values(uint32_t(tid)));
                }
                team_sync<64>();  // learned: the features take the values' place
                if (go) {
                    ch.score(jb.heur, e, dm);
                    if constexpr (LEARN) {
                        if (jb.learn) ch.features(jb, pcode, row, sc, fd);
                    }
                }
                if constexpr (LEARN) {
                    if (jb.learn) {  // uniform; rows of lanes without a child hold what they held
                        team_sync<64>();
                        const uint32_t left = nl - uint32_t(wave) * 32u;
                        const int tiles = __builtin_amdgcn_readfirstlane(left < 32u ? int(left + 7u) / 8 : 4);
                        const float y = forward_wave<nn::Dims<D>::KP>(L.g.net.net, &L.g.net.act[wave][0], tiles, lane);
                        if (go)
                            learned_score<T, D>(y, L.g.net.net.mu, L.g.net.net.sigma, sc, fd, errp, jb.lfloor, pcode, ch.dim, c,
                                                e, dm);
                    }
                }
                if (go) {
                    child_stack(e, bp, b1p, nb, nb1);
#pragma unroll
                    for (int d = 0; d < D; ++d) {
                        const bool cut = d == ch.dim;
                        if (cut && pcode[d] >= 0x80000000u) atomicOr(&L.flags, JF_DEPTH);
                        const uint32_t code = cut ? pcode[d] * 2u + uint32_t(c) : pcode[d];
                        deepest[d] = vmax(deepest[d], 31u - uint32_t(__clz(code)));
                        t.lo[s * D + d] = ch.lo[d];
                        t.hi[s * D + d] = ch.hi[d];
                        t.code[s * D + d] = code;
                    }
                    t.err[s] = e;
                    t.dim[s] = dm;
                    t.b[s] = nb;
                    t.b1[s] = nb1;
                    t.parent[s] = int32_t(node);
                    t.child[s] = -1;
                    t.job[s] = j;
                    if (c == 0) t.child[node] = int32_t(s);
                    pool = nb >= th;
                    atomicAdd(&L.g.hist[grow_place(keys.bucket(nb))], pool ? 0x10001u : 1u);
                }
                const uint32_t k = kept + wave_append(pool, &L.nnew[par]);
                if (pool) {
                    L.g.pool_b[k] = nb;
                    L.g.pool_s[k] = uint32_t(s - base) | uint32_t(dm) << 16;
                }
            }
            count += 2 * nl;
            // the children's stores need not have landed yet: the barrier after the next
            // step's filter orders them before any node of theirs is read
            lds_barrier();
        }
    }
#pragma unroll
    for (int d = 0; d < D; ++d)
        if (deepest[d] != 0) atomicMax(&L.depth[d], deepest[d]);
    __syncthreads();
    if (tid == 0) {
        JobRt& rt = g.rt[j];
        rt.count = base + count;
        rt.flags = L.flags;
        atomicMax(g.rounds + 1, steps);
    }
    if (tid < D && L.depth[tid] != 0) atomicMax(&g.depth[tid], L.depth[tid]);

    if (select) {
        uint32_t n = NONE;
        if (done && jb.N <= GROW_MAX_REGIONS && (need == 0 || L.kb != NONE))
            n = grow_select<T, D, LEARN>(L, t, keys, base, count, need, leaf + jb.reg_base);
        if (n != jb.N)
            for (uint32_t i = tid; i < jb.N; i += NT) leaf[jb.reg_base + i] = -1;
        if (tid == 0) {
            JobRt& rt = g.rt[j];
            rt.nleaves = n == NONE ? 0u : n;
            rt.ties = L.ties;
            if (n == NONE && done && count < need) n = 0;  // too few nodes exist: no route gives N regions
            if (n == NONE) rt.flags |= JF_HANDOVER;
            atomicMax(g.rounds + 6, uint32_t(wall_clock64() - start));
        }
        return;
    }
    // ---- the round kernels' state: the 16-bit histogram of every node, unused slots, and
    // the nodes so far as the first round's candidates (split ones are passed over there)
    {
        uint4* h = reinterpret_cast<uint4*>(g.hist16 + size_t(j) * 65536);
        for (int i = tid; i < 65536 / 4; i += NT) h[i] = make_uint4(0u, 0u, 0u, 0u);
        for (uint32_t i = count + tid; i < jb.node_cap; i += NT) t.job[base + i] = NONE;
        uint32_t* ch = g.defer ? g.chist + size_t(j) * CHIST : nullptr;
        if (ch)
            for (int i = tid; i < CHIST; i += NT) ch[i] = 0;
        __threadfence();  // cleared before any of the block's atomics reach it
        __syncthreads();
        for (uint32_t i = tid; i < count; i += NT) {
            const uint32_t k = key16(t.b[base + i]);
            atomicAdd(&g.hist16[size_t(j) * 65536 + k], 1u);
            if ((k >> 8) != INF_ROW) atomicMax(&L.top_row, k >> 8);
            if (ch && !done && t.child[base + i] < 0) atomicAdd(&ch[k >> 4], 1u);
        }
        __syncthreads();
        if (tid == 0) {
            g.rt[j].row_ceil = L.top_row;
            g.cstart[j] = base;
            g.ncand[j] = done ? 0u : count;
        }
    }
}

}  // namespace vmx

#endif

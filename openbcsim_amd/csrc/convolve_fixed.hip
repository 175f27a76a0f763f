// Convolution and demodulation of one line per workgroup, for transforms of 2^11 to
// 2^14 points and decimations that fold by 1, 2 or 4: conv_line of sim_kernels.hip
// (same spectra, same folds) with every length a constant and the data in place.
//
//   forward   decimation in frequency: a butterfly's outputs go where its inputs were, so
//             that the only barriers are those between passes.  Passes of 16 and 8 points
//             (conv_radix_log2), 16 points a thread; the first reads the line's bins.
//   middle    the last forward pass leaves digit-reversed spectrum samples k0 + m s in one
//             butterfly.  The first inverse pass needs exactly these, and their mirrors
//             N/2 - k, the ones of butterfly m - k0: a thread takes both butterflies and goes
//             from forward outputs over the spectrum (one twiddle for a k and its mirror), its
//             product with H and its folds to inverse inputs in registers.
//   inverse   decimation in time, the forward passes in reverse order; the last one writes
//             the demodulated output.
//
// What bounds it: VALU issue (about 14k wave instructions a line of 2^14 samples, four cycles
// each) and, on top of it rather than beside it, the bins and the IQ: with two workgroups a CU
// the waits of one leave the vector units half idle.  4096 real lines of 9740 samples, folded by
// 2: 148 us, of which 105 without the samples' traffic, 60 for that traffic alone; conv_line,
// whose passes go through LDS to other points and back: 161.  The same with complex bins: 252 (320);
// 2048 lines of 2^13 samples, no fold: 67 (76).  128 of these: 13 (14.2), the chain of one
// wave's instructions.
// Taken back: Stockham passes with the same radices (two barriers a pass, the spectrum through
// LDS: 174 us); padding instead of the mixed slots (conflicts took 0.6 of the LDS cycles);
// workgroups that stay for several lines and load the next one's samples ahead (165 us of 174:
// the loads the last passes wait for queue behind them); delaying every other workgroup (182).
//
// Compiled with -ffp-contract=off; contraction is on inside the transforms.
#include <hip/hip_runtime.h>

#include "fft_math.h"
#include "sim_device.h"

namespace bcsim_hip {

namespace {

template <bool INV>
__device__ __forceinline__ float2 twiddled(float2 a, float2 w) {
#pragma clang fp contract(fast)
    return INV ? make_float2(a.x * w.x + a.y * w.y, a.y * w.x - a.x * w.y) : cmul(a, w);
}

// 16-point DFT: four 4-point DFTs of every fourth input, the sixteenth roots of unity,
// four 4-point DFTs across.  HALF: inputs 8 to 15 are zero and not read.
template <bool INV, bool HALF = false>
__device__ __forceinline__ void dft16(const float2* x, float2* y) {
    constexpr float c1 = 0.92387953251128676f, s1 = 0.38268343236508977f, h = 0.70710678118654752f;
    float2 a[4][4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        if constexpr (HALF) {
            const float2 r = rot90<INV>(x[q + 4]);
            a[q][0] = cadd(x[q], x[q + 4]);
            a[q][1] = cadd(x[q], r);
            a[q][2] = csub(x[q], x[q + 4]);
            a[q][3] = csub(x[q], r);
        } else {
            dft4<INV>(x[q], x[q + 4], x[q + 8], x[q + 12], a[q][0], a[q][1], a[q][2], a[q][3]);
        }
    }
    // a[q][r] *= exp(-2 pi i q r / 16)
    a[1][1] = twiddled<INV>(a[1][1], make_float2(c1, -s1));
    a[1][2] = twiddled<INV>(a[1][2], make_float2(h, -h));
    a[1][3] = twiddled<INV>(a[1][3], make_float2(s1, -c1));
    a[2][1] = twiddled<INV>(a[2][1], make_float2(h, -h));
    a[2][2] = rot90<INV>(a[2][2]);
    a[2][3] = twiddled<INV>(a[2][3], make_float2(-h, -h));
    a[3][1] = twiddled<INV>(a[3][1], make_float2(s1, -c1));
    a[3][2] = twiddled<INV>(a[3][2], make_float2(-h, -h));
    a[3][3] = twiddled<INV>(a[3][3], make_float2(-c1, s1));
#pragma unroll
    for (int r = 0; r < 4; r++) dft4<INV>(a[0][r], a[1][r], a[2][r], a[3][r], y[r], y[r + 4], y[r + 8], y[r + 12]);
}

// a exp(-2 pi i k / 32), 0 <= k < 16
__device__ __forceinline__ float2 turned32(float2 a, int k) {
    constexpr float c[9] = {1.0f,
                            0.98078528040323044f,
                            0.92387953251128676f,
                            0.83146961230254524f,
                            0.70710678118654752f,
                            0.55557023301960222f,
                            0.38268343236508977f,
                            0.19509032201612827f,
                            0.0f};
    if (k == 0) return a;
    if (k == 8) return make_float2(a.y, -a.x);
    return cmul(a, k < 8 ? make_float2(c[k], -c[8 - k]) : make_float2(-c[16 - k], -c[k - 8]));
}

template <int R, bool INV>
__device__ __forceinline__ void dft(const float2* x, float2* y) {
    if constexpr (R == 16) {
        dft16<INV>(x, y);
    } else if constexpr (R == 8) {
        dft8<INV>(x, y);
    } else if constexpr (R == 4) {
        dft4<INV>(x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]);
    } else {
        y[0] = cadd(x[0], x[1]);
        y[1] = csub(x[0], x[1]);
    }
}

// LDS slot of point i of a transform of 2^L points: the low five bits mixed with others, by a
// search over shifts and masks for the ones with the fewest bank conflicts over the accesses of
// all passes here (consecutive points, points 8 or 16 in a row a block apart, the digits of k0).
// Linear over xor: slot(a ^ c) = slot(a) ^ slot(c).
struct Mix {
    int shift[3], mask[3];
};
constexpr Mix kMix[6] = {{{2, 5, 4}, {27, 15, 20}}, {{5, 8, 3}, {29, 27, 24}}, {{4, 9, 8}, {30, 3, 7}},
                         {{3, 4, 9}, {30, 20, 23}}, {{3, 9, 2}, {30, 15, 16}}, {{9, 3, 0}, {30, 25, 0}}};
template <int L>
__host__ __device__ constexpr int slot(int i) {
    constexpr Mix x = kMix[L - 9];
    return i ^ ((i >> x.shift[0]) & x.mask[0]) ^ ((i >> x.shift[1]) & x.mask[1]) ^ ((i >> x.shift[2]) & x.mask[2]);
}

// The point a + C, where C is a constant that shares no bit with a: one xor at most, the rest
// in the instruction's offset.
template <int L>
__device__ __forceinline__ float2& at(float2* buf, int slot_a, int c) {
    const int low = (slot<L>(c) & 31) * 8, high = c & ~31;
    return reinterpret_cast<float2*>(reinterpret_cast<char*>(buf) + ((slot_a * 8) ^ low))[high];
}

// Twiddles w[s - 1] = w^s, 0 < s < R, of a butterfly at column j of a pass's table [R - 1][J].
// Short rows come from the first-level cache.  Of longer ones a thread reads a few and forms
// the others as products: of whole tables a line of 2^14 samples reads 229 KB through the
// second-level cache (4096 lines: 191 us, so 174, with passes as conv_line's).
template <int R, int J>
struct Twiddles {
    static constexpr bool kAll = J < 16;
    float2 w[R - 1];
    __device__ __forceinline__ void load(const float2* __restrict__ tw, int j) {
#pragma unroll
        for (int q = 1; q < R; q++)
            if (kAll || q < 4 || (R == 16 && q % 4 == 0)) w[q - 1] = tw[(q - 1) * J + j];
    }
    __device__ __forceinline__ void complete() {
        if constexpr (!kAll) {
            if constexpr (R == 8) {
                w[3] = cmul(w[1], w[1]);
                w[4] = cmul(w[1], w[2]);
                w[5] = cmul(w[2], w[2]);
                w[6] = cmul(w[2], w[3]);
            } else {
#pragma unroll
                for (int q = 5; q < R; q++)
                    if (q % 4) w[q - 1] = cmul(w[(q & ~3) - 1], w[(q & 3) - 1]);
            }
        }
    }
};

// A pass over the blocks of 2^LB points of a transform of 2^L points, radix 2^RL: butterfly u
// holds the points j + q J of its block (J = 2^(LB - RL), j = u mod J).  Forward: DFT, then
// twiddles; inverse: twiddles, then DFT.  src(u, base, q) and dst(u, base, q, value): the points.
template <int NT, int L, int LB, int RL, bool INV, class Src, class Dst>
__device__ __forceinline__ void pass(const float2* __restrict__ tw, const Src& src, const Dst& dst) {
    constexpr int R = 1 << RL, J = 1 << (LB - RL), B = 1 << (L - RL), IT = (B + NT - 1) / NT;
    const int t = threadIdx.x;
    Twiddles<R, J> w[IT];
    float2 x[IT][R];
#pragma unroll
    for (int it = 0; it < IT; it++) {
        const int u = t + it * NT;
        if (B % NT == 0 || u < B) {
            w[it].load(tw, u & (J - 1));
            const int base = ((u >> (LB - RL)) << LB) + (u & (J - 1));
#pragma unroll
            for (int q = 0; q < R; q++) x[it][q] = src(base, q);
        }
    }
#pragma unroll
    for (int it = 0; it < IT; it++) {
        const int u = t + it * NT;
        if (B % NT == 0 || u < B) {
            const int base = ((u >> (LB - RL)) << LB) + (u & (J - 1));
            w[it].complete();
            float2 y[R];
            if (INV) {
#pragma unroll
                for (int q = 1; q < R; q++) x[it][q] = twiddled<true>(x[it][q], w[it].w[q - 1]);
            }
            dft<R, INV>(x[it], y);
            if (!INV) {
#pragma unroll
                for (int q = 1; q < R; q++) y[q] = cmul(y[q], w[it].w[q - 1]);
            }
#pragma unroll
            for (int q = 0; q < R; q++) dst(base, q, y[q]);
        }
    }
}

// Forward passes I .. before the last one, in place, from blocks of 2^LB points.
template <int NT, int L, int I, int LB>
__device__ __forceinline__ void forward_passes(float2* buf, const float2* __restrict__ roots) {
    constexpr int RL = conv_radix_log2(L, I), J = 1 << (LB - RL);
    if constexpr (I + 1 < conv_passes(L)) {
        pass<NT, L, LB, RL, false>(
            roots + ((1 << L) - (1 << LB)), [buf](int base, int q) { return at<L>(buf, slot<L>(base), q * J); },
            [buf](int base, int q, float2 v) { at<L>(buf, slot<L>(base), q * J) = v; });
        __syncthreads();
        forward_passes<NT, L, I + 1, LB - RL>(buf, roots);
    }
}

// Inverse passes I .. 1, in place, to blocks of 2^LB points (the passes' radices are those of the
// forward transform of 2^LF points); then pass 0 to last(sample, value).
template <int NT, int L, int LF, int I, int LB, class Last>
__device__ __forceinline__ void inverse_passes(float2* buf, const float2* __restrict__ roots, const Last& last) {
    constexpr int RL = conv_radix_log2(LF, I), J = 1 << (LB - RL);
    const float2* tw = roots + ((1 << L) - (1 << LB));
    const auto src = [buf](int base, int q) { return at<L>(buf, slot<L>(base), q * J); };
    if constexpr (I > 0) {
        pass<NT, L, LB, RL, true>(tw, src, [buf](int base, int q, float2 v) { at<L>(buf, slot<L>(base), q * J) = v; });
        __syncthreads();
        inverse_passes<NT, L, LF, I - 1, LB + conv_radix_log2(LF, I - 1)>(buf, roots, last);
    } else {
        pass<NT, L, LB, RL, true>(tw, src, [&](int base, int q, float2 v) { last(base + q * J, v); });
    }
}

// First point of butterfly k0 of the last forward pass (first inverse pass) of a transform of 2^L
// points: the digits of k0 in the forward passes' radices, the first one highest.
template <int L, int LF, int I = 0>
__device__ __forceinline__ int middle_base(int k0) {
    if constexpr (I + 1 < conv_passes(LF)) {
        constexpr int RL = conv_radix_log2(LF, I);
        return ((k0 & ((1 << RL) - 1)) << (L - RL)) + middle_base<L - RL, LF, I + 1>(k0 >> RL);
    } else {
        return 0;
    }
}

// Inverse DFT of the RI inputs v[0 .. N_IN); N_IN = RI / 2: the upper ones are zero but for input
// RI / 2, which is nyquist.
template <int RI, int N_IN>
__device__ __forceinline__ void middle_dft(const float2* v, float2 nyquist, float2* y) {
    if constexpr (N_IN == RI) {
        dft<RI, true>(v, y);
    } else {
        if constexpr (RI == 16) {
            dft16<true, true>(v, y);
        } else {
            float2 x[RI];
#pragma unroll
            for (int i = 0; i < RI; i++) x[i] = i < N_IN ? v[i] : make_float2(0.f, 0.f);
            dft<RI, true>(x, y);
        }
#pragma unroll
        for (int s = 0; s < RI; s++) y[s] = s & 1 ? csub(y[s], nyquist) : cadd(y[s], nyquist);
    }
}

// FULL: complex bins, a transform of N points; else N/2 packed real points.
template <int LOG2N, bool FULL, int FOLD>
__device__ __forceinline__ void conv_fixed_line(const ConvParams& p, int line, float2* buf) {
#pragma clang fp contract(fast)
    constexpr int N = 1 << LOG2N, HALF = N / 2;
    constexpr int L = FULL ? LOG2N : LOG2N - 1;    // forward transform
    constexpr int LM = LOG2N - FOLD;               // inverse transform
    constexpr int NT = conv_fixed_threads(LOG2N, FULL, FOLD);
    constexpr int PASSES = conv_passes(L);
    constexpr int RL = conv_radix_log2(L, PASSES - 1), R = 1 << RL, m = 1 << (L - RL);
    constexpr int RIL = LM - (L - RL), RI = 1 << RIL;
    const int t = threadIdx.x;
    const float2* __restrict__ roots = p.roots;
    const float2* __restrict__ inverse_roots = roots + ((1 << L) - R);
    const float2* __restrict__ H = p.H;

    {
        const int nrf = p.num_rf;
        const float* __restrict__ bins = static_cast<const float*>(p.bins) + (size_t)line * nrf * (FULL ? 2 : 1);
        constexpr int R0 = conv_radix_log2(L, 0), J0 = 1 << (L - R0);
        pass<NT, L, L, R0, false>(
            roots,
            [=](int base, int q) {
                const int i = base + q * J0;
                float2 v = make_float2(0.f, 0.f);
                if (FULL) {
                    if (i < nrf) v = reinterpret_cast<const float2*>(bins)[i];
                } else if (2 * i + 1 < nrf) {
                    __builtin_memcpy(&v, bins + 2 * i, sizeof v);  // lines may start at odd floats
                } else if (2 * i < nrf) {
                    v.x = bins[2 * i];
                }
                return v;
            },
            [buf](int base, int q, float2 v) { at<L>(buf, slot<L>(base), q * J0) = v; });
        __syncthreads();
        forward_passes<NT, L, 1, L - R0>(buf, roots);
    }

    // middle
    const auto points = [&](int k0, float2* y) {
        const int a = slot<L>(middle_base<L, L>(k0));
        float2 x[R];
#pragma unroll
        for (int q = 0; q < R; q++) x[q] = at<L>(buf, a, q);
        dft<R, false>(x, y);
    };
    const auto put = [&](int k0, const float2* y) {
        const int a = slot<LM>(middle_base<LM, L>(k0));
#pragma unroll
        for (int s = 0; s < RI; s++) at<LM>(buf, a, s) = y[s];
    };
    // points written are other points than those read where the lengths differ
    const auto all_read = [] {
        if (LM != L) __syncthreads();
    };
    if constexpr (FULL) {
        constexpr int IT = (m + NT - 1) / NT, USED = R / 2, IN = USED < RI ? USED : RI;
        float2 v[IT][IN], nyquist = make_float2(0.f, 0.f);
#pragma unroll
        for (int it = 0; it < IT; it++) {
            const int k0 = t + it * NT;
            if (m % NT == 0 || k0 < m) {
                float2 z[R];
                points(k0, z);
#pragma unroll
                for (int s = 0; s < USED; s++) {
                    const float2 y = cmul(z[s], H[k0 + m * s]);
                    v[it][s % IN] = s < IN ? y : cadd(v[it][s % IN], y);
                }
                if (k0 == 0) {  // sample N/2
                    nyquist = cmul(z[USED], H[HALF]);
                    if (IN == RI) v[it][0] = cadd(v[it][0], nyquist);
                }
            }
        }
        all_read();
#pragma unroll
        for (int it = 0; it < IT; it++) {
            const int k0 = t + it * NT;
            if (m % NT == 0 || k0 < m) {
                float2 y[RI];
                middle_dft<RI, IN>(v[it], k0 == 0 ? nyquist : make_float2(0.f, 0.f), y);
                put(k0, y);
            }
        }
    } else {
        // Butterflies t and m - t, whose samples mirror one another; thread 0: 0 and m / 2, each
        // its own mirror.  Twice the spectrum: the outputs are halved.
        static_assert(m / 2 <= NT, "a pair of butterflies a thread");
        constexpr int IN = R < RI ? R : RI;
        const int k1 = t ? m - t : m / 2;
        float2 a[R], b[R], nyquist = make_float2(0.f, 0.f);
        if (m / 2 == NT || t < m / 2) {
            points(t, a);
            points(k1, b);
            // X H of k and N/2 - k from the packed transform's samples there; w = exp(-2 pi i k / N)
            const auto spectrum = [=](float2 z, float2 c, float2 w, int root, int k, float2& xk, float2& xm) {
                const float2 e = make_float2(z.x + c.x, z.y - c.y);
                const float2 o = turned32(cmul(make_float2(z.y + c.y, c.x - z.x), w), root);
                xk = cmul(cadd(e, o), H[k]);
                xm = cmul(make_float2(e.x - o.x, o.y - e.y), H[HALF - k]);
            };
            constexpr int TURN = 32 / (2 * R);  // exp(-2 pi i m / N) is a root of order 2 R
            if (t > 0) {
                const float2 w = inverse_roots[(1 << LM) - RI + t];
#pragma unroll
                for (int s = 0; s < R; s++) {
                    const float2 z = a[s], c = b[R - 1 - s];
                    spectrum(z, c, w, s * TURN, t + m * s, a[s], b[R - 1 - s]);
                }
            } else {
                const float2 one = make_float2(1.f, 0.f), w = inverse_roots[(1 << LM) - RI + m / 2];
                float2 unused;
                const float2 z0 = a[0], zm = a[R / 2];
                spectrum(z0, z0, one, 0, 0, a[0], nyquist);
                spectrum(zm, zm, one, R / 2 * TURN, m * (R / 2), a[R / 2], unused);
#pragma unroll
                for (int s = 1; s < R / 2; s++) {
                    const float2 z = a[s], c = a[R - s];
                    spectrum(z, c, one, s * TURN, m * s, a[s], a[R - s]);
                }
#pragma unroll
                for (int s = 0; s < R / 2; s++) {
                    const float2 z = b[s], c = b[R - 1 - s];
                    spectrum(z, c, w, s * TURN, m / 2 + m * s, b[s], b[R - 1 - s]);
                }
            }
#pragma unroll
            for (int s = RI; s < R; s++) {  // folds
                a[s % RI] = cadd(a[s % RI], a[s]);
                b[s % RI] = cadd(b[s % RI], b[s]);
            }
            if (IN == RI) a[0] = cadd(a[0], nyquist);
        }
        all_read();
        if (m / 2 == NT || t < m / 2) {
            float2 y[RI];
            middle_dft<RI, IN>(a, nyquist, y);
            put(t, y);
            middle_dft<RI, IN>(b, make_float2(0.f, 0.f), y);
            put(k1, y);
        }
    }
    __syncthreads();

    // sample E o of the inverse transform is output o
    float2* __restrict__ out = p.iq + (size_t)line * p.n_out;
    const float2* __restrict__ dem = p.demod;
    const int n_out = p.n_out, E = p.out_stride;
    const float scale = FULL ? 1.0f : 0.5f;
    const unsigned inv_e = E > 1 ? 0xffffffffu / (unsigned)E + 1u : 0u;  // i / E = (i inv_e) >> 32 for i < 2^16
    inverse_passes<NT, LM, L, PASSES - 2, RIL + conv_radix_log2(L, PASSES - 2)>(
        buf, inverse_roots, [=](int i, float2 v) {
            int o = i;
            if (E > 1) {
                o = (int)__umulhi((unsigned)i, inv_e);
                if (o * E != i) return;
            }
            if (o < n_out) out[o] = cmul(make_float2(scale * v.x, scale * v.y), dem[o]);
        });
}

template <int LOG2N, bool FULL, int FOLD>
__global__ __launch_bounds__(conv_fixed_threads(LOG2N, FULL, FOLD), 4) void conv_fixed_kernel(ConvParams p) {
    extern __shared__ float2 sbuf[];
    conv_fixed_line<LOG2N, FULL, FOLD>(p, blockIdx.x, sbuf);
}

// One (job, line) pair a workgroup, as convolve_batch_kernel.
template <int LOG2N, bool FULL, int FOLD>
__global__ __launch_bounds__(conv_fixed_threads(LOG2N, FULL, FOLD), 4) void conv_fixed_batch_kernel(
    const ConvParams* __restrict__ jobs, const int2* __restrict__ items) {
    extern __shared__ float2 sbuf[];
    const int2 w = items[blockIdx.x];
    conv_fixed_line<LOG2N, FULL, FOLD>(jobs[w.x], w.y, sbuf);
}

template <int LOG2N, bool FULL, int FOLD>
hipError_t launch(const ConvParams* p, const ConvParams* jobs, const int2* items, int n_items, size_t lds,
                  hipStream_t stream) {
    constexpr int NT = conv_fixed_threads(LOG2N, FULL, FOLD);
    const void* k = p ? (const void*)conv_fixed_kernel<LOG2N, FULL, FOLD>
                      : (const void*)conv_fixed_batch_kernel<LOG2N, FULL, FOLD>;
    hipError_t e = allow_lds(k, lds);
    if (e != hipSuccess) return e;
    if (p) hipLaunchKernelGGL((conv_fixed_kernel<LOG2N, FULL, FOLD>), dim3(p->num_lines), dim3(NT), lds, stream, *p);
    else
        hipLaunchKernelGGL((conv_fixed_batch_kernel<LOG2N, FULL, FOLD>), dim3(n_items), dim3(NT), lds, stream, jobs,
                           items);
    return hipGetLastError();
}

template <int LOG2N, class... A>
hipError_t launch_length(bool full, int fold, A... a) {
    if (full) return fold == 0   ? launch<LOG2N, true, 0>(a...)
                     : fold == 1 ? launch<LOG2N, true, 1>(a...)
                                 : launch<LOG2N, true, 2>(a...);
    return fold == 0   ? launch<LOG2N, false, 0>(a...)
           : fold == 1 ? launch<LOG2N, false, 1>(a...)
                       : launch<LOG2N, false, 2>(a...);
}

template <class... A>
hipError_t launch_any(int log2n, bool full, int fold, A... a) {
    switch (log2n) {
        case 11: return launch_length<11>(full, fold, a...);
        case 12: return launch_length<12>(full, fold, a...);
        case 13: return launch_length<13>(full, fold, a...);
        case 14: return launch_length<14>(full, fold, a...);
    }
    return hipErrorInvalidValue;
}

}  // namespace

hipError_t launch_convolve_fixed(const ConvParams& p, hipStream_t stream) {
    return launch_any(p.log2_len, conv_full(p), p.fold_log2, &p, (const ConvParams*)nullptr, (const int2*)nullptr, 0,
                      conv_lds_bytes(p), stream);
}

hipError_t launch_convolve_fixed_batch(int variant, const ConvParams* jobs, const int2* items, int n_items, size_t lds,
                                       hipStream_t stream) {
    return launch_any(conv_variant_log2(variant), (variant & kConvFull) != 0, conv_variant_fold(variant),
                      (const ConvParams*)nullptr, jobs, items, n_items, lds, stream);
}

}  // namespace bcsim_hip

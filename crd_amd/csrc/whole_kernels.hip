// The long one-kernel transforms of gfx950: n = 2^15 and 2^16 C2C in one launch, each transform held by one
// workgroup from its load to its store.
//
// A CU's register file is 512 KiB and its LDS 160 KiB, so one 512-thread workgroup (256 registers per lane) can keep a
// whole 2^16-point transform (512 KiB): three quarters in registers, a quarter in LDS. The four-step's intermediate
// then never leaves the CU and every point crosses the L2 boundary twice (16 bytes) instead of four times.
//
// n = 256 x N2 (N2 = 32 NT, NT = 4 or 8 column tiles of 32).
//   columns  per tile: thread (lc = tid % 32, li = tid / 32) loads x[(li + 16 m) N2 + 32 tile + lc], m < 16 (runs of
//            256 bytes); a radix-16 pass over m, an exchange through 32 KiB of LDS (real parts, then imaginary parts)
//            that also turns the threads to (i = tid % 16, c = tid / 16), the second radix-16 pass, the four-step
//            twiddle W_n^{col k1} (its table transposed: 128-byte runs). The thread then holds column 32 tile + c at
//            k1 = i + 16 m, again as 16 values, in the registers the tile was loaded into (or, for LT tiles, in LDS
//            slots of its own that no other thread reads).
//   rows     per set of 16 rows (one m, or two of them when NT = 4): 8 values per thread are a register DFT over the
//            tiles; of the 32 points left over c = 4 a + b, a is the wave and b the lane's upper bits: a radix-8 pass
//            over a after an exchange of registers against waves through LDS, a radix-4 pass over b after a swap of
//            registers against lane bits. The 16 rows sit on adjacent lanes, so every store is a run of 128 bytes.
// The registers of a row set are free once it is read, so the next transform's loads go into them at once: they
// are in flight during the rest of the row phase. The grid is at most one workgroup per CU; workgroup b runs transforms
// b, b + grid, ...
//
// Measured (MI355X): n = 2^16 x 2048 0.691 (two four-step passes) -> 0.439 ms, 4.9 TB/s; x 4096 1.39 -> 0.89 ms;
// n = 2^15 x 4096 0.712 -> 0.445 ms, 4.8 TB/s; rel-L2 against FP64 1.45e-7 and 1.39e-7 as before. A round of 256
// transforms of 2^16 takes 55 us against 43 us for its bytes at the copy rate: what is left is the column phase, whose
// LDS exchanges and L2 twiddle reads two waves per SIMD hide only in part.
// What shaped it, at 2^16 x 2048 / 2^15 x 4096: rows kept in lane order through two LDS exchanges per row set 0.615 ms
// / -; the 16 rows on adjacent lanes and one of the exchanges as lane swaps 0.586 / 0.536; each exchange beside the
// arithmetic of the tile or set before and after it, wide exchange spaces 0.548 / 0.498; starts spread within an XCD
// (see launch) 0.490 / 0.445; the twiddles loaded ahead of their products (column_finish) 0.483 / 0.445.
//
// The real transforms of 2^16 reals are the NT = 4 form with the Hermitian recombine inside: C2R pairs each raw tile
// with its mirror through LDS before the column phase (the four-step read every bin twice), R2C pairs each row set's
// outputs with their mirrors through LDS and stores whole 128-byte lines (cross_store). n = 2^16 x 2048: R2C 0.440 ->
// 0.243 ms, C2R 0.451 -> 0.255 ms (4.2-4.4 TB/s); R2C with each run stored as it comes 0.342 ms (a third more bytes
// written: partial lines), the same with non-temporal stores 0.512.
#include "buffer.hpp"
#include "kernels.hpp"

#include <algorithm>

namespace crdfft
{
using namespace dev;

namespace
{

template <int NT> struct WholeCfg
{
    static_assert(NT == 4 || NT == 8, "n = 2^15 or 2^16");
    static constexpr int N1 = 256, N2 = 32 * NT;
    static constexpr uint32_t N = N1 * N2;
    static constexpr int threads = 512;
    static constexpr int LT = NT == 8 ? 2 : 0; // column tiles kept in LDS between the two phases
    static constexpr int ST = NT - LT;         // column tiles kept in registers
    // exchange space from 0. Wide: whole points, 16 rows of 512 at a pitch of 513; NT = 4 alternates between two of
    // them (one barrier each). Narrow: 16 rows of 512 floats at a pitch of 514, real parts then imaginary parts. The
    // pitches put the lanes of one access on different banks. The row exchange takes 8 x 512 points.
    static constexpr int wide_pitch = 513, wide_bytes = 16 * wide_pitch * 8;
    static constexpr int narrow_pitch = 514, narrow_bytes = 16 * narrow_pitch * 4;
    static constexpr bool two_wide = LT == 0;
    // stage twiddles W_256^{i m}, m = 1..15, and W_256^{c q}, q = 1..7
    static constexpr int t1_points = 15 * 16, t2_points = 7 * 32;
    // kept tiles: values of tile S + 1 (all but the last one, which stays in a register) behind the narrow space, over
    // the wide one; those of tile S behind it
    static constexpr int keep1_off = narrow_bytes;
    static constexpr int keep0_off = keep1_off + 15 * threads * 8;
    static constexpr int tab_off = two_wide ? 2 * wide_bytes : keep0_off + 16 * threads * 8;
    static constexpr int lds_bytes = tab_off + (t1_points + t2_points) * 8;
    // real transforms (NT = 4). R2C: the row sets' upper halves cross behind the row exchange's 8 x 512 points of the
    // same wide space; W_n^k1, k1 < 256, follows the tables. C2R: two raw tiles at a pitch of 544 points (512 and the
    // 16 of the tile's or another's first column) and X[h] behind the first one's rows; the tables follow them.
    static constexpr int raw_pitch = 544, raw_bytes = (16 * raw_pitch + 2) * 8;
    static constexpr int cross_off = 8 * threads * 8;
    static_assert(cross_off + 4 * threads * 8 <= wide_bytes, "row exchange and crossing halves");
    static constexpr int r2c_lds_bytes = lds_bytes + 256 * 8;
    static constexpr int c2r_tab_off = 2 * raw_bytes;
    static constexpr int c2r_lds_bytes = c2r_tab_off + (t1_points + t2_points) * 8;
    static_assert(c2r_tab_off >= tab_off || NT != 4, "the C2R tables are clear of both wide spaces");
    static_assert(r2c_lds_bytes <= 160 * 1024 || NT != 4, "LDS of a CU");
    static_assert(c2r_lds_bytes <= 160 * 1024, "LDS of a CU");
    static_assert(narrow_bytes >= 8 * threads * 8, "the row exchange fits the narrow space");
    static_assert(two_wide || keep0_off >= wide_bytes, "the first kept tile is clear of the wide space");
    static_assert(lds_bytes <= 160 * 1024, "LDS of a CU");
};

__device__ __forceinline__ void lane_swap32(float& x, float& y)
{
    const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, y),
                                                    false, false);
    x = __builtin_bit_cast(float, static_cast<uint32_t>(r[0]));
    y = __builtin_bit_cast(float, static_cast<uint32_t>(r[1]));
}

__device__ __forceinline__ void lane_swap16(float& x, float& y)
{
    const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, y),
                                                    false, false);
    x = __builtin_bit_cast(float, static_cast<uint32_t>(r[0]));
    y = __builtin_bit_cast(float, static_cast<uint32_t>(r[1]));
}

// A radix-16 DFT in two halves (the same arithmetic as Dft<16>): four radix-4 DFTs and the inner twiddles, then four
// more. In between, value k1 of the DFT over a[4 n1 + n2] sits at a[4 k1 + n2].
template <bool INV> struct Dft16Halves
{
    template <int N2, int... K1> static __device__ __forceinline__ void twiddle(cf* t, std::integer_sequence<int, K1...>)
    {
        ((t[K1] = twc<static_cast<long>(N2) * K1, 16, INV>(t[K1])), ...);
    }
    template <int N2> static __device__ __forceinline__ void column(cf* a)
    {
        cf t[4] = {a[N2], a[4 + N2], a[8 + N2], a[12 + N2]};
        Dft<4, INV>::run(t);
        twiddle<N2>(t, std::make_integer_sequence<int, 4>{});
#pragma unroll
        for (int k = 0; k < 4; ++k)
        {
            a[4 * k + N2] = t[k];
        }
    }
    static __device__ __forceinline__ void first(cf* a)
    {
        column<0>(a);
        column<1>(a);
        column<2>(a);
        column<3>(a);
    }
    static __device__ __forceinline__ void second(cf* a)
    {
        cf t[16];
#pragma unroll
        for (int k1 = 0; k1 < 4; ++k1)
        {
            cf u[4] = {a[4 * k1], a[4 * k1 + 1], a[4 * k1 + 2], a[4 * k1 + 3]};
            Dft<4, INV>::run(u);
#pragma unroll
            for (int k2 = 0; k2 < 4; ++k2)
            {
                t[k1 + 4 * k2] = u[k2];
            }
        }
#pragma unroll
        for (int k = 0; k < 16; ++k)
        {
            a[k] = t[k];
        }
    }
};

// The segments between two barriers keep their instructions (the scheduler would gather the arithmetic after the last
// barrier and leave the LDS waits bare).
__device__ __forceinline__ void segment_barrier()
{
    __syncthreads();
    __builtin_amdgcn_sched_barrier(0);
}

// The second half of a column tile: v holds the exchanged values (index m of thread i) and leaves with the twiddled X
// at k1 = i + 16 m of column 32 tile + c. The twiddles are on their way during the radix-16 pass, as many as the
// registers hold (loaded one by one where they are used, the phase took twice as long).
template <int NT, bool INV>
__device__ __forceinline__ void column_finish(cf (&v)[16], int tile, const cf* t1, __amdgpu_buffer_rsrc_t tfull)
{
    constexpr int A = NT == 8 ? 8 : 16; // twiddles ahead
    const int tid = threadIdx.x;
    const int i = tid & 15;
    const uint32_t voff = static_cast<uint32_t>(i + 256 * (tid >> 4)) * 8u;
    cf f[16];
#pragma unroll
    for (int m = 0; m < A; ++m)
    {
        f[m] = bld<0>(tfull, voff, static_cast<uint32_t>(16 * m + 256 * 32 * tile) * 8u);
    }
    // stage twiddles: B ahead of their products
    constexpr int B = NT == 8 ? 4 : 15;
    cf g[16];
#pragma unroll
    for (int m = 1; m <= B; ++m)
    {
        g[m] = t1[(m - 1) * 16 + i];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int m0 = 1; m0 < 16; m0 += B)
    {
#pragma unroll
        for (int m = m0; m < m0 + B && m < 16; ++m)
        {
            v[m] = ctw<INV>(v[m], g[m]);
            if (m + B < 16)
            {
                g[m + B] = t1[(m + B - 1) * 16 + i];
            }
        }
        if (m0 + B < 16)
        {
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    Dft<16, INV>::run(v);
    if constexpr (A < 16)
    {
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int m = 0; m < 16; ++m)
    {
        if (m + A < 16)
        {
            f[m + A] = bld<0>(tfull, voff, static_cast<uint32_t>(16 * (m + A) + 256 * 32 * tile) * 8u);
        }
        v[m] = ctw<INV>(v[m], f[m]);
    }
    // the products here, not where they are used: put off, the factors would take registers until then
#pragma unroll
    for (int m = 0; m < 16; ++m)
    {
        asm volatile("" : "+v"(v[m].x), "+v"(v[m].y));
    }
}

// Column phase, tile `v` (after its first radix-16 pass) through the exchange space at `lds` while `fin` finishes the
// tile before it and the next tile's first pass runs in `nx`. TAIL: the space is free for anyone on return.
template <int NT, bool INV, bool WIDE, bool TAIL, bool NEXT, class Fin>
__device__ __forceinline__ void column_exchange(cf (&v)[16], cf (&nx)[16], char* lds, Fin fin)
{
    using C = WholeCfg<NT>;
    const int tid = threadIdx.x;
    if constexpr (WIDE)
    {
        cf* const ex = reinterpret_cast<cf*>(lds);
        cf* const wr = ex + tid;                                            // (k, li, lc) at k pitch + 32 li + lc
        const cf* const rd = ex + (tid & 15) * C::wide_pitch + (tid >> 4);  // (i, m, c)
#pragma unroll
        for (int k = 0; k < 16; ++k)
        {
            wr[k * C::wide_pitch] = v[k];
        }
        fin();
        segment_barrier();
#pragma unroll
        for (int m = 0; m < 16; ++m)
        {
            v[m] = rd[m * 32];
        }
        if constexpr (NEXT)
        {
            Dft16Halves<INV>::first(nx);
            Dft16Halves<INV>::second(nx);
        }
    }
    else
    {
        float* const ex = reinterpret_cast<float*>(lds);
        float* const wr = ex + tid;
        const float* const rd = ex + (tid & 15) * C::narrow_pitch + (tid >> 4);
#pragma unroll
        for (int k = 0; k < 16; ++k)
        {
            wr[k * C::narrow_pitch] = v[k].x;
        }
        fin();
        segment_barrier();
#pragma unroll
        for (int m = 0; m < 16; ++m)
        {
            v[m].x = rd[m * 32];
        }
        if constexpr (NEXT)
        {
            Dft16Halves<INV>::first(nx);
        }
        segment_barrier();
#pragma unroll
        for (int k = 0; k < 16; ++k)
        {
            wr[k * C::narrow_pitch] = v[k].y;
        }
        segment_barrier();
#pragma unroll
        for (int m = 0; m < 16; ++m)
        {
            v[m].y = rd[m * 32];
        }
        if constexpr (NEXT)
        {
            Dft16Halves<INV>::second(nx);
        }
    }
    if constexpr (TAIL)
    {
        segment_barrier();
    }
    else
    {
        __builtin_amdgcn_sched_barrier(0);
    }
}

// KIND of k_whole.
constexpr int kWholeC2C = 0; // x[n] -> X[n], n = 256 N2
constexpr int kWholeR2C = 1; // 2 h reals as z[j] = x[2j] + i x[2j+1] -> X[0 .. h], h = 256 N2 (NT = 4)
constexpr int kWholeC2R = 2; // X[0 .. h] -> 2 h reals, scaled 1 / 2h (NT = 4, INV)

// C2R: Z[j] of one raw tile (c2r_z with scale / 2 in `wa`'s magnitude and `hs`), for row m from X[j] in v[m] and
// X[h - j] at part[(15 - m) raw_pitch]; W_n^j = wa W_2048^{64 m + T}.
template <int T, int M> __device__ __forceinline__ void c2r_point(cf* v, const cf* part, cf wa, float hs)
{
    constexpr int at = (15 - M) * WholeCfg<4>::raw_pitch;
    const cf xk = v[M], xh = part[at];
    const cf w = twc<64 * M + T, 2048, false>(wa);
    const cf e = {(xk.x + xh.x) * hs, (xk.y - xh.y) * hs};
    const cf o = cmulc(cf{xk.x - xh.x, xk.y + xh.y}, w);
    v[M] = cf{e.x - o.y, e.y + o.x};
    asm volatile("" : "+v"(v[M].x), "+v"(v[M].y)); // the value, not its factors, is what waits for the column phase
}
template <int T, int... M>
__device__ __forceinline__ void c2r_tile(cf* v, const cf* part, cf wa, float hs, std::integer_sequence<int, M...>)
{
    (c2r_point<T, M>(v, part, wa, hs), ...);
}

template <int NT, bool INV, int KIND> __global__ __launch_bounds__(512) void k_whole(WholeArgs a)
{
    using C = WholeCfg<NT>;
    constexpr int S = C::ST;
    constexpr int RM = 8 / NT; // values of m per row set
    extern __shared__ __attribute__((aligned(16))) char lds_raw[];
    cf* const keep0 = reinterpret_cast<cf*>(lds_raw + C::keep0_off) + threadIdx.x; // value m at [512 m]
    cf* const keep1 = reinterpret_cast<cf*>(lds_raw + C::keep1_off) + threadIdx.x;
    cf* const t1 = reinterpret_cast<cf*>(lds_raw + (KIND == kWholeC2R ? C::c2r_tab_off : C::tab_off)); // W_256^{i m} at [(m - 1) 16 + i]
    cf* const t2 = t1 + C::t1_points;                           // W_256^{c q} at [(q - 1) 32 + c]
    const int tid = threadIdx.x;
    const int i = tid & 15;
    const int c = tid >> 4;
    const int b = c & 3;
    const int w = tid >> 6; // wave
    {
        const cf* roots = reinterpret_cast<const cf*>(a.roots); // W_256^e
        if (tid < C::t1_points)
        {
            t1[tid] = roots[((tid >> 4) + 1) * (tid & 15)]; // at most 15 * 15
        }
        if (tid < C::t2_points)
        {
            t2[tid] = roots[((tid >> 5) + 1) * (tid & 31)]; // at most 7 * 31
        }
    }
    cf* const wk1 = t2 + C::t2_points; // R2C: W_n^k1
    if constexpr (KIND == kWholeR2C)
    {
        if (tid < 256)
        {
            wk1[tid] = reinterpret_cast<const cf*>(a.wreal)[tid];
        }
    }
    __syncthreads();
    const __amdgpu_buffer_rsrc_t tfull = make_rsrc(a.tfull, C::N * 8u);
    const uint32_t load_off = static_cast<uint32_t>((tid >> 5) * C::N2 + (tid & 31)) * 8u;
    // output i + 16 m + 256 (q + NT s + 8 NT u): wave w holds q = w % NT (of row m0 + w / NT), the lane s = 4 h + b
    const uint32_t store_off = static_cast<uint32_t>(i + 16 * (w / NT) + 256 * (w % NT + NT * b)) * 8u;
    constexpr uint32_t in_bytes = (C::N + (KIND == kWholeC2R ? 1u : 0u)) * 8u;
    constexpr uint32_t out_bytes = (C::N + (KIND == kWholeR2C ? 1u : 0u)) * 8u;
    // C2R rows of h + 1 bins share lines with their neighbours: plain loads
    constexpr int kLoad = KIND == kWholeC2R ? 0 : kAuxNt;

    // R2C (NT = 4): output k = k1 + N1 k2. A set is 16 rows k1 (lanes i) of the lower half in waves 0..3 and their mirrors
    // N1 - k1 in waves 4..7; of a thread's k2, the lower values low + 32 r (r < 4, kStep bins apart) stay and the upper ones
    // low + 16 + 32 r are sent across.
    constexpr int kVal = 4;                           // lower values a thread
    constexpr int kCol = C::N2 / (2 * kVal);          // 16: k2 from a lower value to the upper one after it
    constexpr uint32_t kStep = 2u * kCol * C::N1;     // 8192 bins between a thread's lower values
    static_assert(NT != 4 || (kCol == 16 && kVal * kStep == C::N && C::threads == 512 && RM == 2),
                  "the mirror rules below: 16 rows a set, 4 waves a half, 4 values a thread and half");
    // thread (w, b, i) and its lower values k pair with the upper values, in reverse, of the thread that holds rows -k1:
    // (7 - w, 3 - b, -i); half W_n^{N1 k2} of its lower values
    const int low = (w & 3) + 4 * b;
    const int cross = 64 * (7 - w) + 16 * (3 - b) + ((16 - i) & 15);
    // rows 0 and 128 (lanes i = 0 of the first set) are their own mirrors: k2 -> -k2 and 127 - k2
    const int cross0 = i != 0 ? cross
                              : (w < 4 ? 64 * ((16 - low) & 3) + 16 * (((16 - low) >> 2) & 3) : 64 * (11 - w) + 16 * (3 - b));
    cf wk2[kVal];
    if constexpr (KIND == kWholeR2C)
    {
#pragma unroll
        for (int r = 0; r < kVal; ++r)
        {
            const cf x = reinterpret_cast<const cf*>(a.roots)[low + 2 * kCol * r];
            wk2[r] = cf{0.5f * x.x, 0.5f * x.y};
        }
    }
    // C2R: X[h - j] of the raw tiles 0 .. 3 in their exchange (threads of column 0 find theirs in other tiles)
    const int lc = tid & 31, li = tid >> 5;
    cf* const raw_a = reinterpret_cast<cf*>(lds_raw);
    cf* const raw_b = reinterpret_cast<cf*>(lds_raw + C::raw_bytes);
    const int mirror = 32 * (15 - li) + 32 - lc;
    const cf* const part0 = lc != 0 ? raw_b + mirror : (li != 0 ? raw_a + 32 * (16 - li) : raw_a + C::raw_pitch);
    const cf* const part3 = lc != 0 ? raw_a + mirror : raw_a + 512 + (15 - li);
    const cf* const part1 = lc != 0 ? raw_b + mirror : raw_b + 512 + (15 - li);
    const cf* const part2 = lc != 0 ? raw_a + mirror : raw_b + 32 * (15 - li);
    const float hs = 0.5f / static_cast<float>(C::N);
    cf wa{};
    if constexpr (KIND == kWholeC2R)
    {
        const cf x = reinterpret_cast<const cf*>(a.wreal)[li * C::N2 + lc];
        wa = cf{hs * x.x, hs * x.y};
    }

    for (uint32_t d = ((blockIdx.x >> 3) & 31u) * a.stagger; d > 0; --d)
    {
        __builtin_amdgcn_s_sleep(16); // 1024 clocks
    }
    uint64_t t = blockIdx.x;
    cf s[S][16];
    cf last{}; // NT = 8: value 15 of the second kept tile; C2R: X[h] (in thread 0)
    // slots S - LT + l first hold the LDS tiles (numbers S + l), then their own
    {
        const __amdgpu_buffer_rsrc_t src = make_rsrc(reinterpret_cast<const cf*>(a.in) + t * a.idist, in_bytes);
#pragma unroll
        for (int m = 0; m < 16; ++m)
        {
#pragma unroll
            for (int q = 0; q < S; ++q)
            {
                const int tile = q < S - C::LT ? q : q + C::LT;
                s[q][m] = bld<kLoad>(src, load_off, static_cast<uint32_t>(16 * m * C::N2 + 32 * tile) * 8u);
            }
        }
        if constexpr (KIND == kWholeC2R)
        {
            last = bld<kLoad>(src, C::N * 8u, 0);
        }
    }
#pragma unroll 1
    for (; t < a.count; t += gridDim.x)
    {
        const __amdgpu_buffer_rsrc_t src = make_rsrc(reinterpret_cast<const cf*>(a.in) + t * a.idist, in_bytes);
        if constexpr (KIND == kWholeC2R)
        {
            // raw tiles 0 and 3, then 1 and 2, against their mirrors
            constexpr auto rows = std::make_integer_sequence<int, 16>{};
            // through an empty asm: the 64 products with wa are not to be kept in registers across transforms
            asm volatile("" : "+v"(wa.x), "+v"(wa.y));
            segment_barrier(); // the row exchange of the transform before is read
#pragma unroll
            for (int m = 0; m < 16; ++m)
            {
                raw_a[m * C::raw_pitch + tid] = s[0][m];
                raw_b[m * C::raw_pitch + tid] = s[3][m];
            }
            if (lc == 0)
            {
#pragma unroll
                for (int m = 0; m < 16; ++m)
                {
                    raw_a[m * C::raw_pitch + 512 + li] = s[1][m];
                    raw_b[m * C::raw_pitch + 512 + li] = s[3][m];
                }
            }
            if (tid == 0)
            {
                raw_a[16 * C::raw_pitch] = last;
            }
            segment_barrier();
            c2r_tile<0>(s[0], part0, wa, hs, rows);
            c2r_tile<3>(s[3], part3, wa, hs, rows);
            segment_barrier();
#pragma unroll
            for (int m = 0; m < 16; ++m)
            {
                raw_a[m * C::raw_pitch + tid] = s[1][m];
                raw_b[m * C::raw_pitch + tid] = s[2][m];
            }
            segment_barrier();
            c2r_tile<1>(s[1], part1, wa, hs, rows);
            c2r_tile<2>(s[2], part2, wa, hs, rows);
            segment_barrier();
        }
        if constexpr (C::LT > 0)
        {
            // column phase: tile 6 (kept in LDS) from slot 4, tiles 0-2, tile 7 (kept) from slot 5, tile 3, then tiles
            // 4 and 5, loaded into slots 4 and 5 as soon as those are free. The wide space is there until tile 7 is
            // kept.
            static_assert(NT == 8 && S == 6, "the order below");
            auto reload = [&](int q) {
#pragma unroll
                for (int m = 0; m < 16; ++m)
                {
                    s[q][m] = bld<kAuxNt>(src, load_off, static_cast<uint32_t>(16 * m * C::N2 + 32 * q) * 8u);
                }
            };
            Dft<16, INV>::run(s[4]);
            column_exchange<NT, INV, true, true, true>(s[4], s[0], lds_raw, [] {});
            column_exchange<NT, INV, true, true, true>(s[0], s[1], lds_raw, [&] {
                column_finish<NT, INV>(s[4], 6, t1, tfull);
#pragma unroll
                for (int m = 0; m < 16; ++m)
                {
                    keep0[m * C::threads] = s[4][m];
                }
                reload(4);
            });
            column_exchange<NT, INV, true, true, true>(s[1], s[2], lds_raw,
                                                       [&] { column_finish<NT, INV>(s[0], 0, t1, tfull); });
            column_exchange<NT, INV, true, true, true>(s[2], s[5], lds_raw,
                                                       [&] { column_finish<NT, INV>(s[1], 1, t1, tfull); });
            column_exchange<NT, INV, true, true, true>(s[5], s[3], lds_raw,
                                                       [&] { column_finish<NT, INV>(s[2], 2, t1, tfull); });
            column_exchange<NT, INV, false, true, true>(s[3], s[4], lds_raw, [&] {
                column_finish<NT, INV>(s[5], 7, t1, tfull);
#pragma unroll
                for (int m = 0; m < 15; ++m)
                {
                    keep1[m * C::threads] = s[5][m];
                }
                last = s[5][15];
                reload(5);
            });
            column_exchange<NT, INV, false, true, true>(s[4], s[5], lds_raw,
                                                        [&] { column_finish<NT, INV>(s[3], 3, t1, tfull); });
            column_exchange<NT, INV, false, true, false>(s[5], s[5], lds_raw,
                                                         [&] { column_finish<NT, INV>(s[4], 4, t1, tfull); });
            column_finish<NT, INV>(s[5], 5, t1, tfull);
        }
        else
        {
            // column phase: tiles 0 .. S - 1, alternating between the two wide spaces
            Dft<16, INV>::run(s[0]);
            column_exchange<NT, INV, true, false, true>(s[0], s[1], lds_raw, [] {});
#pragma unroll
            for (int q = 1; q < S; ++q)
            {
                char* const space = lds_raw + (q & 1) * C::wide_bytes;
                auto fin = [&] { column_finish<NT, INV>(s[q - 1], q - 1, t1, tfull); };
                if (q + 1 < S)
                {
                    column_exchange<NT, INV, true, false, true>(s[q], s[q + 1 < S ? q + 1 : q], space, fin);
                }
                else
                {
                    column_exchange<NT, INV, true, false, false>(s[q], s[q], space, fin);
                }
            }
            column_finish<NT, INV>(s[S - 1], S - 1, t1, tfull);
        }
        // the next transform of this workgroup (no records when there is none: its loads return zeros)
        const bool more = t + gridDim.x < a.count;
        const __amdgpu_buffer_rsrc_t nsrc =
            make_rsrc(reinterpret_cast<const cf*>(a.in) + (more ? t + gridDim.x : t) * a.idist, more ? in_bytes : 0u);
        const __amdgpu_buffer_rsrc_t dst = make_rsrc(reinterpret_cast<cf*>(a.out) + t * a.odist, out_bytes);
        cf u[8], y[8];
        constexpr int kSets = 16 / RM;
        // row set j: m = j (NT = 8), 2 j and 2 j + 1 (NT = 4), or for R2C j and its mirror 15 - j, so that every row
        // -k1 is in the set; the mirrors of the rows i = 0 are one m further on (m = 0 and 8 mirror themselves and
        // share the first set)
        auto rows_first = [&](int j) {
#pragma unroll
            for (int mm = 0; mm < RM; ++mm)
            {
                const int m0 = KIND == kWholeR2C ? (mm == 0 ? j : 15 - j) : RM * j + mm;
#pragma unroll
                for (int q = 0; q < S; ++q)
                {
                    u[mm * NT + q] = s[q][m0];
                    if (KIND == kWholeR2C && mm == 1)
                    {
                        const cf z = s[q][j == 0 ? 8 : 16 - j];
                        u[mm * NT + q].x = i == 0 ? z.x : u[mm * NT + q].x;
                        u[mm * NT + q].y = i == 0 ? z.y : u[mm * NT + q].y;
                    }
                }
                if constexpr (C::LT > 0)
                {
                    u[S] = keep0[m0 * C::threads];
                    u[S + 1] = m0 < 15 ? keep1[m0 * C::threads] : last;
                }
                Dft<NT, INV>::run(u + mm * NT);
#pragma unroll
                for (int q = 1; q < NT; ++q)
                {
                    u[mm * NT + q] = ctw<INV>(u[mm * NT + q], t2[(q * (8 / NT) - 1) * 32 + c]); // W_N2^{c q}
                }
            }
        };
        // the next transform's points for the registers that no set after j reads
        auto prefetch_row = [&](int m) {
#pragma unroll
            for (int q = 0; q < S; ++q)
            {
                const int tile = q < S - C::LT ? q : q + C::LT;
                s[q][m] = bld<kLoad>(nsrc, load_off, static_cast<uint32_t>(16 * m * C::N2 + 32 * tile) * 8u);
            }
        };
        auto prefetch = [&](int j) {
            if (KIND != kWholeR2C)
            {
#pragma unroll
                for (int mm = 0; mm < RM; ++mm)
                {
                    prefetch_row(RM * j + mm);
                }
                return;
            }
            prefetch_row(j);
            if (j > 0)
            {
                prefetch_row(16 - j);
            }
            if (j == kSets - 1)
            {
                prefetch_row(8);
            }
        };
        // a row set after its exchange (in y): the last two passes; y[4 h + e] is then the output of
        // k2 = q + NT (4 h + b) + 8 NT e
        auto rows_last = [&] {
            Dft<8, INV>::run(y);
#pragma unroll
            for (int e = 1; e < 8; ++e)
            {
                y[e] = ctw<INV>(y[e], t2[(e - 1) * 32 + 8 * b]); // W_32^{b e}
            }
            // the low two bits of s (registers) <-> b (lane bits 4 and 5)
#pragma unroll
            for (int e = 0; e < 8; ++e)
            {
                if ((e & 2) == 0)
                {
                    lane_swap32(y[e].x, y[e + 2].x);
                    lane_swap32(y[e].y, y[e + 2].y);
                }
            }
#pragma unroll
            for (int e = 0; e < 8; e += 2)
            {
                lane_swap16(y[e].x, y[e + 1].x);
                lane_swap16(y[e].y, y[e + 1].y);
            }
            Dft<4, INV>::run(y);
            Dft<4, INV>::run(y + 4);
        };
        auto store = [&](int j) {
#pragma unroll
            for (int h = 0; h < 2; ++h)
            {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                {
                    const cf o = {y[h * 4 + e].x * a.scale, y[h * 4 + e].y * a.scale};
                    bst<kAuxNt>(dst, store_off, static_cast<uint32_t>(16 * RM * j + 256 * (4 * NT * h + 8 * NT * e)) * 8u,
                                o);
                }
            }
        };
        // R2C: the upper values go to their mirrors' threads, the lower ones stay (z)
        cf z[4];
        auto cross_write = [&](int j) {
            cf* const x = reinterpret_cast<cf*>(lds_raw + (j & 1) * C::wide_bytes + C::cross_off) + tid;
#pragma unroll
            for (int r = 0; r < 4; ++r)
            {
                z[r] = y[r];
                x[r * 512] = y[4 + r];
            }
        };
        // X[k] = E + W_n^k O and X[h-k] = conj(E - W_n^k O), E = (z + conj p) / 2, O = (z - conj p) / 2i, p = Z[h-k]
        // (real_fft.hpp:41-68)
        auto mirror_pair = [](cf zk, cf p, cf wk, cf& xk, cf& xh) {
            const cf e = {(zk.x + p.x) * 0.5f, (zk.y - p.y) * 0.5f};
            const cf o = cmul(cf{zk.y + p.y, p.x - zk.x}, wk);
            xk = cadd(e, o);
            xh = cf{e.x - o.x, o.y - e.y};
        };
        // A set's 16 rows are runs of 16 bins, which start anywhere in a 128-byte line (h + 1 bins a transform): the
        // lanes past the end of the line the run shares with the set before store that set's value, so a store
        // instruction writes whole lines. Residue of lane i in its line: sg + i for the lower rows' k (w < 4, runs
        // moving up by 16 a set) and the upper rows' (moving down), sg - i for their mirrors.
        const uint32_t sg =
            static_cast<uint32_t>((reinterpret_cast<uintptr_t>(a.out) >> 3) + t * a.odist) & 15u;
        const uint32_t res = (sg + i) & 15u, res_h = (sg - i) & 15u;
        const bool now = w < 4 ? res >= sg : res < ((sg + 1) & 15u);
        const bool now_h = w < 4 ? res_h < ((sg + 1) & 15u) : res_h >= sg;
        // from a set's address back to the one before: rows 16 lower (w < 4) or higher
        const uint32_t back = now ? 0u : (w < 4 ? 0u - 128u : 128u);
        const uint32_t back_h = now_h ? 0u : (w < 4 ? 128u : 0u - 128u);
        const bool odd_row = i == 0 && w >= 4; // row N1 / 2 in the first set, not row N1
        constexpr uint32_t kFar = 0x40000000u; // outside the resource: dropped
        cf old[4], old_h[4];
        auto cross_store = [&](int j) {
            const cf* const x = reinterpret_cast<const cf*>(lds_raw + (j & 1) * C::wide_bytes + C::cross_off);
            // through an empty asm, so that the addresses of all sets are not kept in registers across transforms
            int iv = i, lowv = low;
            asm volatile("" : "+v"(iv), "+v"(lowv));
            // lower waves: rows i + 16 j; upper waves: rows i + N1 - 16 (j + 1), but for i = 0, whose lower row 16 j mirrors to
            // N1 - 16 j, one set on (row N1 / 2 in the first set: rows 0 and N1 / 2 are their own mirrors)
            constexpr int kTop = C::N1 - 16;
            const int k1 = w < 4 ? iv + 16 * j : iv + kTop - 16 * j + (iv == 0 ? (j == 0 ? C::N1 / 2 - kTop : 16) : 0);
            const cf wk = wk1[k1];
            const uint32_t k = static_cast<uint32_t>(k1 + C::N1 * lowv); // k + kStep r
            uint32_t at = k * 8u, at_h = (C::N - k - (kVal - 1) * kStep) * 8u;
            cf p[4];
#pragma unroll
            for (int r = 0; r < 4; ++r)
            {
                p[r] = x[(3 - r) * 512 + (j == 0 ? cross0 : cross)];
            }
            if (j == 0)
            {
                // in thread 0 k = kStep r mirrors within the thread, and so do its upper values k = kMid + kStep r (the other
                // threads' stores of those are dropped)
                constexpr uint32_t kMid = static_cast<uint32_t>(kCol * C::N1), kMid1 = kMid + kStep;
                const bool t0 = tid == 0;
#pragma unroll
                for (int r = 0; r < 4; ++r)
                {
                    const cf o = z[(4 - r) & 3];
                    p[r] = cf{t0 ? o.x : p[r].x, t0 ? o.y : p[r].y};
                }
                const uint32_t far = t0 ? 0u : kFar;
                cf xk, xh;
                mirror_pair(x[0], x[3 * 512], cf{0.5f * W<kCol, C::N1>::re, 0.5f * W<kCol, C::N1>::im}, xk, xh);
                bst<0>(dst, far, kMid * 8u, xk);
                bst<0>(dst, far, (C::N - kMid) * 8u, xh);
                mirror_pair(x[512], x[2 * 512], cf{0.5f * W<3 * kCol, C::N1>::re, 0.5f * W<3 * kCol, C::N1>::im}, xk, xh);
                bst<0>(dst, far, kMid1 * 8u, xk);
                bst<0>(dst, far, (C::N - kMid1) * 8u, xh);
                at = now || odd_row ? at : kFar;
                at_h = now_h || odd_row ? at_h : kFar;
            }
            else
            {
                at = j == 1 && odd_row && !now ? kFar : at + back;
                at_h = j == 1 && odd_row && !now_h ? kFar : at_h + back_h;
            }
#pragma unroll
            for (int r = 0; r < 4; ++r)
            {
                cf xk, xh;
                mirror_pair(z[r], p[r], cmul(wk, wk2[r]), xk, xh);
                if (j == 0 && r == 0)
                {
                    // X[0] and X[h] without their products (exact, but for an infinity times the zero parts)
                    xk = tid == 0 ? cf{z[0].x + z[0].y, 0.0f} : xk;
                    xh = tid == 0 ? cf{z[0].x - z[0].y, 0.0f} : xh;
                }
                const uint32_t step = kStep * 8u * static_cast<uint32_t>(r), step_h = kStep * 8u * static_cast<uint32_t>(kVal - 1 - r);
                if (j == 0)
                {
                    bst<0>(dst, at, step, xk);
                    bst<0>(dst, at_h, step_h, xh);
                }
                else
                {
                    bst<kAuxNt>(dst, at, step, cf{now ? xk.x : old[r].x, now ? xk.y : old[r].y});
                    bst<kAuxNt>(dst, at_h, step_h, cf{now_h ? xh.x : old_h[r].x, now_h ? xh.y : old_h[r].y});
                }
                old[r] = xk;
                old_h[r] = xh;
            }
            if (j == kSets - 1)
            {
                // what the last set left for a line that no set follows
                at = now ? kFar : k * 8u;
                at_h = now_h ? kFar : (C::N - k - (kVal - 1) * kStep) * 8u;
#pragma unroll
                for (int r = 0; r < 4; ++r)
                {
                    bst<0>(dst, at, kStep * 8u * static_cast<uint32_t>(r), old[r]);
                    bst<0>(dst, at_h, kStep * 8u * static_cast<uint32_t>(kVal - 1 - r), old_h[r]);
                }
            }
        };
        rows_first(0);
#pragma unroll
        for (int j = 0; j < kSets; ++j)
        {
            // register r of wave w <-> register w of wave r; the set before finishes beside the writes, the set after
            // starts beside the reads
            cf* const exc = reinterpret_cast<cf*>(lds_raw + (C::two_wide ? (j & 1) * C::wide_bytes : 0));
#pragma unroll
            for (int r = 0; r < 8; ++r)
            {
                exc[r * 512 + tid] = u[r];
            }
            prefetch(j);
            if (j > 0)
            {
                rows_last();
                if constexpr (KIND == kWholeR2C)
                {
                    cross_write(j - 1);
                }
                else
                {
                    store(j - 1);
                }
            }
            segment_barrier();
#pragma unroll
            for (int e = 0; e < 8; ++e)
            {
                y[e] = exc[w * 512 + e * 64 + (tid & 63)];
            }
            if constexpr (KIND == kWholeR2C)
            {
                if (j > 0)
                {
                    cross_store(j - 1);
                }
            }
            if (j + 1 < kSets)
            {
                rows_first(j + 1);
            }
            if constexpr (C::two_wide)
            {
                __builtin_amdgcn_sched_barrier(0);
            }
            else
            {
                segment_barrier();
            }
        }
        rows_last();
        if constexpr (KIND == kWholeR2C)
        {
            cross_write(kSets - 1);
            segment_barrier();
            cross_store(kSets - 1);
        }
        else
        {
            store(kSets - 1);
        }
        if constexpr (KIND == kWholeC2R)
        {
            last = bld<kLoad>(nsrc, C::N * 8u, 0);
        }
    }
}

// The start of the workgroups of an XCD is spread over 31 * stagger * 1024 clocks: in step, all CUs load and store in
// the row phase at once and leave the memory idle in the column phase.
template <int NT, bool INV, int KIND> hipError_t launch(WholeArgs a, unsigned grid, hipStream_t s)
{
    const uint64_t rounds = a.count / grid;
    a.stagger = NT == 8 ? (rounds >= 4 ? 2u : 1u) : (rounds >= 4 ? 1u : 0u);

    using C = WholeCfg<NT>;
    auto kern = k_whole<NT, INV, KIND>;
    constexpr int lds = KIND == kWholeR2C ? C::r2c_lds_bytes : (KIND == kWholeC2R ? C::c2r_lds_bytes : C::lds_bytes);
    const hipError_t e =
        hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess)
    {
        return e;
    }
    hipLaunchKernelGGL(kern, dim3(grid), dim3(C::threads), lds, s, a);
    return hipGetLastError();
}

} // namespace

bool whole_kernel_n(uint64_t n, uint64_t* n2)
{
    if (n != WholeCfg<4>::N && n != WholeCfg<8>::N)
    {
        return false;
    }
    *n2 = n / 256;
    return true;
}

hipError_t launch_whole(uint64_t n, bool inverse, const WholeArgs& a, unsigned grid, hipStream_t s)
{
    if (a.count == 0)
    {
        return hipSuccess;
    }
    grid = static_cast<unsigned>(std::min<uint64_t>(grid, a.count));

    if (grid == 0 || a.tfull == nullptr || a.roots == nullptr)
    {
        return hipErrorInvalidValue;
    }
    if (n == WholeCfg<4>::N)
    {
        return inverse ? launch<4, true, kWholeC2C>(a, grid, s) : launch<4, false, kWholeC2C>(a, grid, s);
    }
    if (n == WholeCfg<8>::N)
    {
        return inverse ? launch<8, true, kWholeC2C>(a, grid, s) : launch<8, false, kWholeC2C>(a, grid, s);
    }
    return hipErrorInvalidValue;
}

hipError_t launch_whole_real(uint64_t h, bool c2r, const WholeArgs& a, unsigned grid, hipStream_t s)
{
    if (a.count == 0)
    {
        return hipSuccess;
    }
    grid = static_cast<unsigned>(std::min<uint64_t>(grid, a.count));
    if (grid == 0 || h != WholeCfg<4>::N || a.tfull == nullptr || a.roots == nullptr || a.wreal == nullptr)
    {
        return hipErrorInvalidValue;
    }
    return c2r ? launch<4, true, kWholeC2R>(a, grid, s) : launch<4, false, kWholeR2C>(a, grid, s);
}

} // namespace crdfft

// gfx950 kernels for the per-rank data path: element-wise reduce / copy over descriptor tables.
// Bandwidth-bound work: 128-bit coalesced loads and stores, several independent loads in flight per
// lane, no LDS, no matrix cores.  One launch covers every step of a phase (or every fused item) for
// all ranks; a workgroup walks tiles of kTileBytes with a grid stride.
//
// Arithmetic rules (must match bit for bit on every path):
//   integers   sum / prod wrap modulo 2^n; max = (b > a) ? b : a, min = (b < a) ? b : a
//   fp32/fp64  one IEEE operation per combine, same max / min selection rule
//   fp16/bf16  widen to fp32, combine, round to nearest even; max / min keep the chosen operand's bits
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

#include "kernels.h"

namespace hcclamd {

typedef uint32_t V4 __attribute__((ext_vector_type(4)));   // 16 bytes, one global_load_dwordx4

struct HalfBits { uint16_t v; };
struct Bf16Bits { uint16_t v; };

enum : int { ROP_SUM = 0, ROP_PROD = 1, ROP_MAX = 2, ROP_MIN = 3 };

// ---- element arithmetic ---------------------------------------------------------------------------
template <typename T> struct UnsignedOf { using type = T; };
template <> struct UnsignedOf<int8_t> { using type = uint8_t; };
template <> struct UnsignedOf<int16_t> { using type = uint16_t; };
template <> struct UnsignedOf<int32_t> { using type = uint32_t; };
template <> struct UnsignedOf<int64_t> { using type = uint64_t; };

template <typename T, int OP> struct Elem {
    // integers
    static __device__ __forceinline__ T Apply(T a, T b)
    {
        using U = typename UnsignedOf<T>::type;
        if (OP == ROP_SUM) {
            return static_cast<T>(static_cast<U>(static_cast<uint32_t>(static_cast<U>(a)) + static_cast<uint32_t>(static_cast<U>(b))));
        } else if (OP == ROP_PROD) {
            return static_cast<T>(static_cast<U>(static_cast<uint32_t>(static_cast<U>(a)) * static_cast<uint32_t>(static_cast<U>(b))));
        } else if (OP == ROP_MAX) {
            return (b > a) ? b : a;
        } else {
            return (b < a) ? b : a;
        }
    }
};
template <typename T, int OP> struct Elem64 {
    static __device__ __forceinline__ T Apply(T a, T b)
    {
        if (OP == ROP_SUM) {
            return static_cast<T>(static_cast<uint64_t>(a) + static_cast<uint64_t>(b));
        } else if (OP == ROP_PROD) {
            return static_cast<T>(static_cast<uint64_t>(a) * static_cast<uint64_t>(b));
        } else if (OP == ROP_MAX) {
            return (b > a) ? b : a;
        } else {
            return (b < a) ? b : a;
        }
    }
};
template <int OP> struct Elem<int64_t, OP> : Elem64<int64_t, OP> {};
template <int OP> struct Elem<uint64_t, OP> : Elem64<uint64_t, OP> {};

template <typename F, int OP> struct ElemFloat {
    static __device__ __forceinline__ F Apply(F a, F b)
    {
        if (OP == ROP_SUM) {
            return a + b;
        } else if (OP == ROP_PROD) {
            return a * b;
        } else if (OP == ROP_MAX) {
            return (b > a) ? b : a;
        } else {
            return (b < a) ? b : a;
        }
    }
};
template <int OP> struct Elem<float, OP> : ElemFloat<float, OP> {};
template <int OP> struct Elem<double, OP> : ElemFloat<double, OP> {};

__device__ __forceinline__ float Bf16ToFloat(uint16_t b) { return __uint_as_float(static_cast<uint32_t>(b) << 16); }
__device__ __forceinline__ uint16_t FloatToBf16(float f)
{
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) {
        return static_cast<uint16_t>((u >> 16) | 0x0040u);
    }
    u += 0x7fffu + ((u >> 16) & 1u);
    return static_cast<uint16_t>(u >> 16);
}
__device__ __forceinline__ float HalfToFloat(uint16_t h)
{
    _Float16 x;
    __builtin_memcpy(&x, &h, 2);
    return static_cast<float>(x);
}
__device__ __forceinline__ uint16_t FloatToHalf(float f)
{
    _Float16 x = static_cast<_Float16>(f);   // v_cvt_f16_f32, round to nearest even
    uint16_t h;
    __builtin_memcpy(&h, &x, 2);
    return h;
}

template <int OP> struct Elem<HalfBits, OP> {
    static __device__ __forceinline__ HalfBits Apply(HalfBits a, HalfBits b)
    {
        float fa = HalfToFloat(a.v), fb = HalfToFloat(b.v);
        HalfBits r;
        if (OP == ROP_SUM) {
            r.v = FloatToHalf(fa + fb);
        } else if (OP == ROP_PROD) {
            r.v = FloatToHalf(fa * fb);
        } else if (OP == ROP_MAX) {
            r.v = (fb > fa) ? b.v : a.v;
        } else {
            r.v = (fb < fa) ? b.v : a.v;
        }
        return r;
    }
};
template <int OP> struct Elem<Bf16Bits, OP> {
    static __device__ __forceinline__ Bf16Bits Apply(Bf16Bits a, Bf16Bits b)
    {
        float fa = Bf16ToFloat(a.v), fb = Bf16ToFloat(b.v);
        Bf16Bits r;
        if (OP == ROP_SUM) {
            r.v = FloatToBf16(fa + fb);
        } else if (OP == ROP_PROD) {
            r.v = FloatToBf16(fa * fb);
        } else if (OP == ROP_MAX) {
            r.v = (fb > fa) ? b.v : a.v;
        } else {
            r.v = (fb < fa) ? b.v : a.v;
        }
        return r;
    }
};

// 16 bytes of T combined lane by lane; a is the rank's own operand, b the peer's.
template <typename T, int OP> struct Combiner {
    static __device__ __forceinline__ V4 Apply(V4 a, V4 b)
    {
        constexpr int N = 16 / sizeof(T);
        union U {
            V4 v;
            T e[N];
            __device__ U() {}
        } ua, ub, ur;
        ua.v = a;
        ub.v = b;
#pragma unroll
        for (int i = 0; i < N; i++) {
            ur.e[i] = Elem<T, OP>::Apply(ua.e[i], ub.e[i]);
        }
        return ur.v;
    }
};

// Narrow types work on whole 32-bit words with packed 16-bit instructions (v_pk_*_u16 / _i16) and the
// hardware bf16 conversion (v_cvt_pk_bf16_f32, round to nearest even), a fraction of the instructions
// that element-by-element extraction costs; the results are the same bits.
typedef short S2 __attribute__((ext_vector_type(2)));
typedef unsigned short U2 __attribute__((ext_vector_type(2)));
typedef float F2 __attribute__((ext_vector_type(2)));
typedef __bf16 B2 __attribute__((ext_vector_type(2)));

template <typename To, typename From> __device__ __forceinline__ To BitCast(From f)
{
    static_assert(sizeof(To) == sizeof(From), "size");
    To t;
    __builtin_memcpy(&t, &f, sizeof(To));
    return t;
}

template <bool SIGNED, int OP> __device__ __forceinline__ uint32_t Pk16(uint32_t a, uint32_t b)
{
    if (OP == ROP_SUM) {
        return BitCast<uint32_t>(U2(BitCast<U2>(a) + BitCast<U2>(b)));
    } else if (OP == ROP_PROD) {
        return BitCast<uint32_t>(U2(BitCast<U2>(a) * BitCast<U2>(b)));
    } else if (SIGNED) {
        S2 x = BitCast<S2>(a), y = BitCast<S2>(b);
        return BitCast<uint32_t>(OP == ROP_MAX ? __builtin_elementwise_max(x, y) : __builtin_elementwise_min(x, y));
    } else {
        U2 x = BitCast<U2>(a), y = BitCast<U2>(b);
        return BitCast<uint32_t>(OP == ROP_MAX ? __builtin_elementwise_max(x, y) : __builtin_elementwise_min(x, y));
    }
}

template <bool SIGNED, int OP> __device__ __forceinline__ uint32_t Pk8(uint32_t a, uint32_t b)
{
    if (OP == ROP_SUM) {
        // add the low 7 bits of every byte, then fix the top bits without carrying across bytes
        return ((a & 0x7f7f7f7fu) + (b & 0x7f7f7f7fu)) ^ ((a ^ b) & 0x80808080u);
    } else if (OP == ROP_PROD) {
        uint32_t even = Pk16<false, ROP_PROD>(a & 0x00ff00ffu, b & 0x00ff00ffu) & 0x00ff00ffu;
        uint32_t odd = Pk16<false, ROP_PROD>((a >> 8) & 0x00ff00ffu, (b >> 8) & 0x00ff00ffu) & 0x00ff00ffu;
        return even | (odd << 8);
    } else {
        // a byte moved to the top of a 16-bit lane compares like the byte itself
        uint32_t even = Pk16<SIGNED, OP>((a << 8) & 0xff00ff00u, (b << 8) & 0xff00ff00u);
        uint32_t odd = Pk16<SIGNED, OP>(a & 0xff00ff00u, b & 0xff00ff00u);
        return ((even >> 8) & 0x00ff00ffu) | odd;
    }
}

template <int OP> __device__ __forceinline__ uint32_t PkBf16(uint32_t a, uint32_t b)
{
    const uint32_t aLo = a << 16, aHi = a & 0xffff0000u, bLo = b << 16, bHi = b & 0xffff0000u;
    const float faLo = __uint_as_float(aLo), faHi = __uint_as_float(aHi);
    const float fbLo = __uint_as_float(bLo), fbHi = __uint_as_float(bHi);
    if (OP == ROP_SUM || OP == ROP_PROD) {
        F2 r;
        r.x = (OP == ROP_SUM) ? faLo + fbLo : faLo * fbLo;
        r.y = (OP == ROP_SUM) ? faHi + fbHi : faHi * fbHi;
        return BitCast<uint32_t>(__builtin_convertvector(r, B2));
    } else {
        const bool pickLo = (OP == ROP_MAX) ? (fbLo > faLo) : (fbLo < faLo);
        const bool pickHi = (OP == ROP_MAX) ? (fbHi > faHi) : (fbHi < faHi);
        return ((pickHi ? bHi : aHi)) | ((pickLo ? bLo : aLo) >> 16);
    }
}

// fp16, two elements per word.  Sum and product use the packed half instructions (v_pk_add_f16 / v_pk_mul_f16), one
// per word instead of four conversions, two operations and a conversion back.  The bits are those of "widen to fp32,
// combine, round to nearest even": an fp32 has 24 significant bits, 2 x 11 + 2, and with that many the second rounding
// of a sum never changes what a single rounding to 11 bits gives (the product of two halves is exact in fp32 to begin
// with); denormal halves are kept by both forms.  Max / min compare the halves as they are (the conversion to fp32 is
// exact and keeps the order) and keep the chosen operand's bits.
typedef _Float16 H2 __attribute__((ext_vector_type(2)));
template <int OP> __device__ __forceinline__ uint32_t PkF16(uint32_t a, uint32_t b)
{
    const H2 x = BitCast<H2>(a), y = BitCast<H2>(b);
    if (OP == ROP_SUM || OP == ROP_PROD) {
        const H2 r = (OP == ROP_SUM) ? x + y : x * y;
        return BitCast<uint32_t>(r);
    } else {
        const bool pickLo = (OP == ROP_MAX) ? (y.x > x.x) : (y.x < x.x);
        const bool pickHi = (OP == ROP_MAX) ? (y.y > x.y) : (y.y < x.y);
        return ((pickHi ? b : a) & 0xffff0000u) | ((pickLo ? b : a) & 0x0000ffffu);
    }
}

#define HCCL_WORDWISE_COMBINER(TYPE, EXPR)                                  \
    template <int OP> struct Combiner<TYPE, OP> {                           \
        static __device__ __forceinline__ V4 Apply(V4 a, V4 b)              \
        {                                                                   \
            V4 r;                                                           \
            r.x = EXPR(a.x, b.x);                                           \
            r.y = EXPR(a.y, b.y);                                           \
            r.z = EXPR(a.z, b.z);                                           \
            r.w = EXPR(a.w, b.w);                                           \
            return r;                                                       \
        }                                                                   \
    };
#define HCCL_EXPR_I16(x, y) Pk16<true, OP>(x, y)
#define HCCL_EXPR_U16(x, y) Pk16<false, OP>(x, y)
#define HCCL_EXPR_I8(x, y) Pk8<true, OP>(x, y)
#define HCCL_EXPR_U8(x, y) Pk8<false, OP>(x, y)
#define HCCL_EXPR_BF16(x, y) PkBf16<OP>(x, y)
#define HCCL_EXPR_F16(x, y) PkF16<OP>(x, y)
HCCL_WORDWISE_COMBINER(int16_t, HCCL_EXPR_I16)
HCCL_WORDWISE_COMBINER(uint16_t, HCCL_EXPR_U16)
HCCL_WORDWISE_COMBINER(int8_t, HCCL_EXPR_I8)
HCCL_WORDWISE_COMBINER(uint8_t, HCCL_EXPR_U8)
HCCL_WORDWISE_COMBINER(Bf16Bits, HCCL_EXPR_BF16)
HCCL_WORDWISE_COMBINER(HalfBits, HCCL_EXPR_F16)

template <typename T, int OP> __device__ __forceinline__ V4 Combine16(V4 a, V4 b) { return Combiner<T, OP>::Apply(a, b); }

// ---- memory access ---------------------------------------------------------------------------------
// 16 bytes at an address of any alignment: the device runs in unaligned-access mode, so this is still
// one 128-bit load or store (one that may touch two memory lines).
typedef uint32_t V4U __attribute__((ext_vector_type(4), aligned(1)));

// Rank buffers are device (global) memory.  The pointers come out of descriptor tables, so the
// compiler cannot know that and would issue flat accesses, whose completion is counted together
// with scalar loads (a wait for the next descriptor pointer then also waits for every load in
// flight).  Casting to the global address space gives global_load / global_store.
#define HCCL_GLOBAL __attribute__((address_space(1)))
typedef V4 HCCL_GLOBAL GlobalV4;
typedef V4U HCCL_GLOBAL GlobalV4U;

// 16 bytes in LDS (the gather kernel's staging area; the tiles a team kernel holds between its read and write phases)
typedef V4 __attribute__((address_space(3))) LdsV4;
typedef V4U __attribute__((address_space(3))) LdsV4U;

template <uint32_t MODE> __device__ __forceinline__ V4 Load16(const void *base, uint64_t byteOff)
{
    const char *p = static_cast<const char *>(base) + byteOff;
    if (MODE == ACC_VEC16) {
        return __builtin_nontemporal_load((const GlobalV4 *)p);
    } else {
        V4U t = __builtin_nontemporal_load((const GlobalV4U *)p);
        return V4{t.x, t.y, t.z, t.w};
    }
}
// 16 bytes at any address, fetched as whole words: the four words from the word boundary in front on, and the word that
// holds the last bytes (for an address on a word boundary the fourth word again, so that nothing outside the words of
// the 16 bytes is touched; the words at a block's ends hold up to three bytes before and behind it, which may lie outside the
// caller's buffer: they are read with their word, never past it, and dropped).  Vector(shift) puts them together, shift =
// address mod 4.
// For 8-bit elements: a 128-bit load off a word boundary costs the vector memory unit more than the extra word does.
// Reduce-scatter, int8, blocks of odd length, us, 128-bit loads / this way: 8 ranks x 3 000 017 sum 44.2 / 42.1 (blocks at
// multiples of 64 bytes: 39.9), x 12 000 017 168.0 / 157.5; 16 ranks x 700 001 sum 47.1 / 43.1, max 55.6 / 47.2.  16-bit
// elements gain nothing (bf16 sum 8 x 1 000 001 30.5 / 31.1, fp16 8 x 2 000 001 51.6 / 52.2) and keep the 128-bit loads.
struct WordVec {
    V4 v;
    uint32_t last;
    __device__ __forceinline__ void Load(const void *base, uint64_t byteOff, uint32_t shift)
    {
        typedef uint32_t HCCL_GLOBAL GlobalWord;
        typedef uint32_t V4W __attribute__((ext_vector_type(4), aligned(4)));
        typedef V4W HCCL_GLOBAL GlobalV4W;
        const char *p = static_cast<const char *>(base) - shift + byteOff;
        const V4W t = __builtin_nontemporal_load((const GlobalV4W *)p);
        v = V4{t.x, t.y, t.z, t.w};
        last = *(const GlobalWord *)(p + (shift != 0 ? 16 : 12));
    }
    __device__ __forceinline__ V4 Vector(uint32_t shift) const
    {
        return V4{__builtin_amdgcn_alignbyte(v.y, v.x, shift), __builtin_amdgcn_alignbyte(v.z, v.y, shift),
            __builtin_amdgcn_alignbyte(v.w, v.z, shift), __builtin_amdgcn_alignbyte(last, v.w, shift)};
    }
};
__device__ __forceinline__ void Store16(void *base, uint64_t byteOff, V4 v)
{
    __builtin_nontemporal_store(v, (GlobalV4 *)(static_cast<char *>(base) + byteOff));
}

// 16 bytes at an address of any alignment, past the caches.
__device__ __forceinline__ void StoreAny16(void *base, uint64_t pos, V4 v)
{
    V4U t = {v.x, v.y, v.z, v.w};
    __builtin_nontemporal_store(t, (GlobalV4U *)(static_cast<char *>(base) + pos));
}

// Stores through a buffer descriptor: a choice of cache policies that plain stores do not have, one descriptor per
// destination and tile instead of an address per lane and vector, and whatever lies at or behind its `bytes` is dropped.  The
// address need not be aligned.  Policies, MI355X, plain streaming kernels, TB/s read and written (non-temporal alone /
// ordinary / through / through + non-temporal):
//   8 sources, 8 destinations of 4, 12, 24, 96 MiB   6.1 / 5.7 / 6.3 / 6.2   5.6 / - / 5.8 / 5.6   5.6 / 5.3 / 5.6 / 5.6   5.5 / 5.4 / 5.5 / 5.6
//   1 source, 8 destinations of 4, 24, 96 MiB        5.2 / 4.8 / 6.1 / 5.9   5.4 / 5.1 / 5.5 / 5.5   5.2 / 5.1 / 5.3 / 5.2
//   8 sources, 1 destination of 8, 32, 48, 96 MiB    6.1 / - / 6.2 / 6.1   6.3 / - / 6.5 / 6.1   6.3 / - / 6.5 / 6.2   6.1 / - / 6.1 / 6.1
//   one to one, 32, 96 MiB                           5.3 / - / 5.9 / 5.5   6.0 / - / 6.2 / 6.1
// Which one: StoreFlags (launch_rules.h) for the plain kernels; the team kernels stream unless the caller has set otherwise.
enum StorePolicy : uint32_t {
    STORE_ORDINARY = 0,      // write-back
    STORE_NT = 2,            // non-temporal
    STORE_THROUGH = 16,      // past the L2 at once, kept in the memory-side cache
    STORE_STREAMED = 18      // both
};
typedef __amdgpu_buffer_rsrc_t BufferRsrc;
__device__ __forceinline__ BufferRsrc MakeBuffer(void *base, uint32_t bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(base, 0, int(bytes), 0x00020000);
}
template <uint32_t POLICY> __device__ __forceinline__ void BufferStore16(BufferRsrc r, uint32_t pos, V4 v)
{
    __builtin_amdgcn_raw_buffer_store_b128(v, r, int(pos), 0, int(POLICY));
}

// Element-wise access to global memory (heads, tails, unaligned buffers).
template <size_t N> struct ElemCarrier;
template <> struct ElemCarrier<1> { typedef uint8_t type; };
template <> struct ElemCarrier<2> { typedef uint16_t type; };
template <> struct ElemCarrier<4> { typedef uint32_t type; };
template <> struct ElemCarrier<8> { typedef uint64_t type; };
template <typename T> __device__ __forceinline__ T LoadElem(const void *base, uint64_t byteOff)
{
    typedef typename ElemCarrier<sizeof(T)>::type C;
    C c = *(const C HCCL_GLOBAL *)(static_cast<const char *>(base) + byteOff);
    T t;
    __builtin_memcpy(&t, &c, sizeof(T));
    return t;
}
template <typename T> __device__ __forceinline__ void StoreElem(void *base, uint64_t byteOff, T t)
{
    typedef typename ElemCarrier<sizeof(T)>::type C;
    C c;
    __builtin_memcpy(&c, &t, sizeof(T));
    *(C HCCL_GLOBAL *)(static_cast<char *>(base) + byteOff) = c;
}

// Accesses of the step kernel.  Loads are non-temporal; stores are ordinary write-back stores: what
// one phase writes the next phase reads, and part of it is still in the memory-side cache then
// (measured, 8-rank fp32 ring all-reduce of 256 MiB per rank, 14 phases: 1.478 ms with non-temporal
// stores, 1.433 ms with ordinary ones; ordinary loads instead cost 9 %).  The fused kernels write
// results nobody reads back (StorePolicy; ordinary stores cost them 7 % at 256 MiB per rank).
__device__ __forceinline__ V4 StepLoad(const void *base, uint64_t byteOff)
{
    return Load16<ACC_VEC16>(base, byteOff);
}
template <bool ORDINARY> __device__ __forceinline__ void StepStore(void *base, uint64_t byteOff, V4 v)
{
    if (ORDINARY) {
        *(GlobalV4 *)(static_cast<char *>(base) + byteOff) = v;
    } else {
        Store16(base, byteOff, v);
    }
}

// Largest i with table[i].tile0 <= tile (tile0 is ascending, table[0].tile0 == 0).
template <typename D> __device__ __forceinline__ uint32_t FindDesc(const D *table, uint32_t n, uint32_t tile)
{
    uint32_t lo = 0, hi = n;
    while (hi - lo > 1) {
        uint32_t mid = (lo + hi) >> 1;
        if (table[mid].tile0 <= tile) {
            lo = mid;
        } else {
            hi = mid;
        }
    }
    return lo;
}

// Item of a tile in a fused launch.  When every item of the launch covers `tilesPerItem` tiles (the last one at most
// as many; 0 = they differ), the index follows from the tile number and the table search, a chain of dependent loads
// that is most of a small collective's time, is not needed.
template <typename D> __device__ __forceinline__ uint32_t ItemOfTile(const D *table, uint32_t n, uint32_t tile, uint32_t tilesPerItem)
{
    if (tilesPerItem != 0) {
        const uint32_t i = tile / tilesPerItem;
        return i < n ? i : n - 1;
    }
    return FindDesc(table, n, tile);
}

constexpr uint32_t kVecPerLane = kTileBytes / (kBlockThreads * 16);   // 4

// ---- one phase of copy / reduce steps -----------------------------------------------------------------
template <typename T, int OP, uint32_t MODE>
__device__ __forceinline__ void StepTileVec(const StepDesc &d, uint64_t off, uint32_t n)
{
    const uint32_t nvec = n >> 4;
    const uint32_t tid = threadIdx.x;
    if (nvec == kTileBytes / 16) {
        V4 va[kVecPerLane], vb[kVecPerLane];
#pragma unroll
        for (uint32_t u = 0; u < kVecPerLane; u++) {
            va[u] = Load16<MODE>(d.a, off + (uint64_t(u) * kBlockThreads + tid) * 16);
        }
        if (d.b != nullptr) {
#pragma unroll
            for (uint32_t u = 0; u < kVecPerLane; u++) {
                vb[u] = Load16<MODE>(d.b, off + (uint64_t(u) * kBlockThreads + tid) * 16);
            }
#pragma unroll
            for (uint32_t u = 0; u < kVecPerLane; u++) {
                va[u] = Combine16<T, OP>(va[u], vb[u]);
            }
        }
#pragma unroll
        for (uint32_t u = 0; u < kVecPerLane; u++) {
            Store16(d.dst, off + (uint64_t(u) * kBlockThreads + tid) * 16, va[u]);
        }
    } else {
        for (uint32_t i = tid; i < nvec; i += kBlockThreads) {
            V4 v = Load16<MODE>(d.a, off + uint64_t(i) * 16);
            if (d.b != nullptr) {
                v = Combine16<T, OP>(v, Load16<MODE>(d.b, off + uint64_t(i) * 16));
            }
            Store16(d.dst, off + uint64_t(i) * 16, v);
        }
    }
}

template <typename T, int OP>
__device__ __forceinline__ void StepTileElem(const StepDesc &d, uint64_t off, uint32_t n)
{
    const uint32_t cnt = n / sizeof(T);
    for (uint32_t i = threadIdx.x; i < cnt; i += kBlockThreads) {
        const uint64_t at = off + uint64_t(i) * sizeof(T);
        T v = LoadElem<T>(d.a, at);
        if (d.b != nullptr) {
            v = Elem<T, OP>::Apply(v, LoadElem<T>(d.b, at));
        }
        StoreElem<T>(d.dst, at, v);
    }
}

// Fast loop of the step kernel over tiles [blockIdx.x, nwhole) with stride gridDim.x: every tile is
// whole and ACC_VEC16.  The descriptor of the next tile is looked up while the loads of the current
// one are in flight (the lookup is a chain of dependent scalar loads), and not at all while the next
// tile still belongs to the current step.  ORDINARY picks the store kind at compile time (a run-time
// choice per store is folded into one store by the compiler).
template <typename T, int OP, bool ORDINARY>
__device__ __forceinline__ void StepWholeTiles(const StepDesc *__restrict__ steps, uint32_t nsteps, uint32_t nwhole, uint32_t ntiles,
    bool reverse)
{
    const uint32_t tid = threadIdx.x;
    uint32_t tile = blockIdx.x;
    uint32_t idx = FindDesc(steps, nsteps, tile);
    StepDesc d = steps[idx];
    uint32_t dEnd = idx + 1 < nsteps ? steps[idx + 1].tile0 : ntiles;   // first tile past this step
    for (;;) {
        // whole tiles only, so walking a step backwards is a matter of the index
        const uint64_t off = uint64_t(reverse ? dEnd - 1 - tile : tile - d.tile0) * kTileBytes;
        const uint32_t next = tile + gridDim.x;
        const bool reduce = d.b != nullptr;
        V4 va[kVecPerLane], vb[kVecPerLane];
#pragma unroll
        for (uint32_t u = 0; u < kVecPerLane; u++) {
            va[u] = StepLoad(d.a, off + (uint64_t(u) * kBlockThreads + tid) * 16);
        }
        if (reduce) {
#pragma unroll
            for (uint32_t u = 0; u < kVecPerLane; u++) {
                vb[u] = StepLoad(d.b, off + (uint64_t(u) * kBlockThreads + tid) * 16);
            }
        }
        // keep the loads above where they are: without this the compiler sinks them below the lookup
        asm volatile("" ::: "memory");
        StepDesc dn = d;
        uint32_t dnEnd = dEnd;
        if (next < nwhole && next >= dEnd) {
            idx = FindDesc(steps, nsteps, next);
            dn = steps[idx];
            dnEnd = idx + 1 < nsteps ? steps[idx + 1].tile0 : ntiles;
        }
        if (reduce) {
#pragma unroll
            for (uint32_t u = 0; u < kVecPerLane; u++) {
                va[u] = Combine16<T, OP>(va[u], vb[u]);
            }
        }
#pragma unroll
        for (uint32_t u = 0; u < kVecPerLane; u++) {
            StepStore<ORDINARY>(d.dst, off + (uint64_t(u) * kBlockThreads + tid) * 16, va[u]);
        }
        if (next >= nwhole) {
            break;
        }
        tile = next;
        d = dn;
        dEnd = dnEnd;
    }
}

// Tiles [0, nwhole) belong to steps that are ACC_VEC16 and a whole number of tiles (the host puts
// those first in the table); tiles [nwhole, ntiles) are everything else: ragged ends, unaligned
// buffers.  The two get separate loops: with the slow paths in the same loop as the fast one, the
// compiler's wait-count bookkeeping (which joins all paths at the loop head) makes every iteration
// wait for the previous iteration's stores before it issues its loads.
template <typename T, int OP>
__global__ void __launch_bounds__(kBlockThreads) StepKernel(const StepDesc *__restrict__ steps, uint32_t nsteps, uint32_t nwhole,
    uint32_t ntiles, uint32_t flags)
{
    if (blockIdx.x < nwhole) {
        if (flags & kStepOrdinaryStores) {
            StepWholeTiles<T, OP, true>(steps, nsteps, nwhole, ntiles, (flags & kStepReverse) != 0);
        } else {
            StepWholeTiles<T, OP, false>(steps, nsteps, nwhole, ntiles, (flags & kStepReverse) != 0);
        }
    }
    for (uint32_t tile = nwhole + blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const StepDesc d = steps[FindDesc(steps, nsteps, tile)];
        const uint64_t off = uint64_t(tile - d.tile0) * kTileBytes;
        const uint64_t left = d.bytes - off;
        const uint32_t n = left < kTileBytes ? uint32_t(left) : kTileBytes;
        if (d.mode == ACC_VEC16) {
            StepTileVec<T, OP, ACC_VEC16>(d, off, n);
        } else if (d.mode == ACC_VEC16_ANY) {
            StepTileVec<T, OP, ACC_VEC16_ANY>(d, off, n);
        } else {
            StepTileElem<T, OP>(d, off, n);
        }
    }
}

// ---- fused kernels: what they share ---------------------------------------------------------------------
// The tiles of a launch come in three parts.  Tiles [0, nwhole) are whole: they belong to the first nitems items.  Then comes a
// tile for the rest of every item's body (of an item with less than a tile all of it), then one for every item's ends.  The loop over whole tiles has
// nothing else in it: with the guarded paths in the same loop the compiler makes a tile's loads wait for each other and for
// the stores of the tile before.  Rests and ends go through the same straight-line code, all sources' loads in flight: one
// after the other they were most of a ragged collective of a few MiB (all-reduce, 8 ranks, bf16, 2 MiB + 6 bytes per rank
// 20.9 us, now 8.0; 32 ranks 77.6, now 27.9).
constexpr uint32_t kChainVec = 4;      // vectors per lane per pass

// Operand order changes the bits only where the combine is not commutative bit for bit:
// floating max / min (NaN and signed zero follow the selection rule).
template <typename T, int OP> struct OrderMatters { static constexpr bool value = false; };
template <int OP> struct OrderMatters<float, OP> { static constexpr bool value = (OP == ROP_MAX || OP == ROP_MIN); };
template <int OP> struct OrderMatters<double, OP> { static constexpr bool value = (OP == ROP_MAX || OP == ROP_MIN); };
template <int OP> struct OrderMatters<HalfBits, OP> { static constexpr bool value = (OP == ROP_MAX || OP == ROP_MIN); };
template <int OP> struct OrderMatters<Bf16Bits, OP> { static constexpr bool value = (OP == ROP_MAX || OP == ROP_MIN); };

// What a lane works on: 16 bytes, or one element.  `base` is the same for the whole wave, `pos` a lane's offset from it.
// What is loaded is a Raw; Value makes a Val of it.  Accesses are unaligned ones (the instruction is the same one), so one
// form serves every alignment.
template <typename T, int OP> struct VecLane {
    typedef V4 Val;
    typedef V4 Raw;
    typedef V4 Out;
    typedef VecLane Exact;
    static constexpr bool kChecked = false;      // Combine gives the same bits as Elem for every operand
    static constexpr bool kHoldBack = sizeof(T) == 1 && OP == ROP_SUM;      // see TreeFold
    static __device__ __forceinline__ Out Result(const Val &v) { return v; }
    static __device__ __forceinline__ Raw Load(const void *base, uint32_t pos) { return Load16<ACC_VEC16_ANY>(base, pos); }
    static __device__ __forceinline__ Val Value(const Raw &r, const void *) { return r; }
    static __device__ __forceinline__ void Store(void *base, uint32_t pos, Val v) { StoreAny16(base, pos, v); }
    static __device__ __forceinline__ Val Combine(Val a, Val b) { return Combine16<T, OP>(a, b); }
};
template <typename T, int OP> struct WordLane {
    typedef V4 Val;
    typedef WordVec Raw;
    typedef V4 Out;
    typedef WordLane Exact;
    static constexpr bool kChecked = false;
    static __device__ __forceinline__ Out Result(const Val &v) { return v; }
    static __device__ __forceinline__ uint32_t Shift(const void *base) { return uint32_t(reinterpret_cast<uintptr_t>(base)) & 3u; }
    static __device__ __forceinline__ Raw Load(const void *base, uint32_t pos)
    {
        Raw r;
        r.Load(base, pos, Shift(base));
        return r;
    }
    static __device__ __forceinline__ Val Value(const Raw &r, const void *base) { return r.Vector(Shift(base)); }
    static __device__ __forceinline__ Val Combine(Val a, Val b) { return Combine16<T, OP>(a, b); }
};
template <typename T, int OP> struct ElemLane {
    typedef T Val;
    typedef T Raw;
    typedef T Out;
    typedef ElemLane Exact;
    static constexpr bool kChecked = false;
    static constexpr bool kHoldBack = false;
    static __device__ __forceinline__ Out Result(const Val &v) { return v; }
    static __device__ __forceinline__ Raw Load(const void *base, uint32_t pos) { return LoadElem<T>(base, pos); }
    static __device__ __forceinline__ Val Value(const Raw &r, const void *) { return r; }
    static __device__ __forceinline__ void Store(void *base, uint32_t pos, Val v) { StoreElem<T>(base, pos, v); }
    static __device__ __forceinline__ Val Combine(Val a, Val b) { return Elem<T, OP>::Apply(a, b); }
};

// How a chain folds 16 bytes: 8-bit types always, 16-bit max / min where all loads of up to 8 sources are in flight (with more
// sources, or two sources at a time, they take Exact).  Most types: VecLane.  Where a combine takes several instructions per word because elements have
// to be taken apart and put together again, the value is kept apart from the first source to the last (instructions per word and
// source: 8-bit 3 instead of 6 to 11; bf16 max / min 3 or 2 instead of 9; fp16 max / min 1 or half a one instead of 5).
template <typename T, int OP> struct FoldLane : VecLane<T, OP> {};

struct SplitVec { V4 a, b; };

// 8-bit: the even and the odd bytes each in 16-bit lanes.  Sum and product only look at the low byte of a lane, max and min
// are decided by the high byte: what else a lane holds does not matter, so nothing is masked.
template <bool SIGNED, int OP> struct ByteLane {
    typedef SplitVec Val;
    typedef V4 Raw;
    typedef V4 Out;
    typedef ByteLane Exact;
    static constexpr bool kChecked = false;
    static constexpr bool kHigh = OP == ROP_MAX || OP == ROP_MIN;
    static __device__ __forceinline__ Raw Load(const void *base, uint32_t pos) { return Load16<ACC_VEC16_ANY>(base, pos); }
    static __device__ __forceinline__ Val Value(const Raw &r, const void *) { return kHigh ? Val{r << 8, r} : Val{r, r >> 8}; }
    static __device__ __forceinline__ V4 Each(V4 x, V4 y)
    {
        return V4{Pk16<SIGNED, OP>(x.x, y.x), Pk16<SIGNED, OP>(x.y, y.y), Pk16<SIGNED, OP>(x.z, y.z), Pk16<SIGNED, OP>(x.w, y.w)};
    }
    static __device__ __forceinline__ Val Combine(const Val &x, const Val &y) { return Val{Each(x.a, y.a), Each(x.b, y.b)}; }
    static __device__ __forceinline__ uint32_t Join(uint32_t even, uint32_t odd)
    {
        // bytes of the first operand are 4 ... 7 of the selector, of the second 0 ... 3
        return kHigh ? __builtin_amdgcn_perm(odd, even, 0x07030501u) : __builtin_amdgcn_perm(odd, even, 0x06020400u);
    }
    static __device__ __forceinline__ Out Result(const Val &v)
    {
        return V4{Join(v.a.x, v.b.x), Join(v.a.y, v.b.y), Join(v.a.z, v.b.z), Join(v.a.w, v.b.w)};
    }
};
template <int OP> struct FoldLane<int8_t, OP> : ByteLane<true, OP> {};
template <int OP> struct FoldLane<uint8_t, OP> : ByteLane<false, OP> {};

// Max / min of 16-bit floats by the instructions that hand a NaN on (v_maximum3 / v_minimum3).  The selection rule
// ((b > a) ? b : a in the schedule's order) gives the same bits unless a source is a NaN, and the result then is one, or the result
// is a zero and sources are zeros of both signs, between which the rule goes by the order.  Of these the instructions take +0 for a
// maximum and -0 for a minimum: a zero result of the other sign is right as it is, and this one where no source holds the other.
// ChainWhole looks at the first source, then at the result, then at all sources, still in registers, and folds by the rule where it has to.
// All-reduce, 8 ranks, bf16 maximum, us, always by the rule / folded again for every zero or NaN / this way: 64 MiB normal data
// 196 / 177 / 177, 1 % zeros 198 / 199 / 182, negative values as zeros 197 / 202 / 183, zeros of both signs 196 / 203 / 188, 1 % NaNs 197 / 202 / 188, one
// NaN in 1200 results 197 / 199 / 200; 2 MiB 8.7 / 6.3 / 6.3, 8.8 / 8.8 / 7.0, 8.9 / 9.1 / 7.3, 8.6 / 9.0 / 8.7, 8.6 / 8.9 / 8.3, 8.6 / 8.7 / 9.0; fp16 64 MiB 187 / 173 /
// 176, 188 / 185 / 181, 189 / 193 / 182, 188 / 192 / 182, 189 / 192 / 183, 189 / 187 / 191.
template <uint32_t INF, int OP> struct SpecialHalves {
    uint32_t most = 0, least = ~0u, leastSigned = 0x7fff7fffu;
    // NaNs, and zeros of either sign: the largest of (magnitude - 1) per half is not below INF then
    __device__ __forceinline__ void SeeAny(V4 v)
    {
#pragma unroll
        for (uint32_t i = 0; i < 4; i++) {
            most = BitCast<uint32_t>(__builtin_elementwise_max(BitCast<U2>(most), BitCast<U2>(v[i] & 0x7fff7fffu) - U2{1, 1}));
        }
    }
    __device__ __forceinline__ bool Any() const { return (most & 0xffffu) >= INF || (most >> 16) >= INF; }
    // NaNs: the largest magnitude is above INF
    __device__ __forceinline__ void SeeNan(V4 v)
    {
#pragma unroll
        for (uint32_t i = 0; i < 4; i++) {
            most = BitCast<uint32_t>(__builtin_elementwise_max(BitCast<U2>(most), BitCast<U2>(v[i] & 0x7fff7fffu)));
        }
    }
    __device__ __forceinline__ bool Nan() const { return (most & 0xffffu) > INF || (most >> 16) > INF; }
    // +0 is the least number without sign, -0 the least with one
    __device__ __forceinline__ void SeePlus(V4 v)
    {
#pragma unroll
        for (uint32_t i = 0; i < 4; i++) {
            least = BitCast<uint32_t>(__builtin_elementwise_min(BitCast<U2>(least), BitCast<U2>(v[i])));
        }
    }
    __device__ __forceinline__ bool Plus() const { return (least & 0xffffu) == 0 || (least >> 16) == 0; }
    __device__ __forceinline__ void SeeMinus(V4 v)
    {
#pragma unroll
        for (uint32_t i = 0; i < 4; i++) {
            leastSigned = BitCast<uint32_t>(__builtin_elementwise_min(BitCast<S2>(leastSigned), BitCast<S2>(v[i])));
        }
    }
    __device__ __forceinline__ bool Minus() const { return (leastSigned & 0xffffu) == 0x8000u || (leastSigned >> 16) == 0x8000u; }
    // the zero that the instructions take, and the one that they pass over
    __device__ __forceinline__ void SeeTaken(V4 v) { OP == ROP_MAX ? SeePlus(v) : SeeMinus(v); }
    __device__ __forceinline__ bool Taken() const { return OP == ROP_MAX ? Plus() : Minus(); }
    __device__ __forceinline__ void SeePassed(V4 v) { OP == ROP_MAX ? SeeMinus(v) : SeePlus(v); }
    __device__ __forceinline__ bool Passed() const { return OP == ROP_MAX ? Minus() : Plus(); }
};
template <int OP> struct HalfMaxLane {
    typedef V4 Val;
    typedef V4 Raw;
    typedef V4 Out;
    typedef VecLane<HalfBits, OP> Exact;
    typedef SpecialHalves<0x7c00u, OP> Special;
    static constexpr bool kChecked = true;
    static __device__ __forceinline__ Raw Load(const void *base, uint32_t pos) { return Load16<ACC_VEC16_ANY>(base, pos); }
    static __device__ __forceinline__ Val Value(const Raw &r, const void *) { return r; }
    static __device__ __forceinline__ uint32_t Each(uint32_t x, uint32_t y)
    {
        const H2 a = BitCast<H2>(x), b = BitCast<H2>(y);
        return BitCast<uint32_t>(OP == ROP_MAX ? __builtin_elementwise_maximum(a, b) : __builtin_elementwise_minimum(a, b));
    }
    static __device__ __forceinline__ Val Combine(V4 x, V4 y) { return V4{Each(x.x, y.x), Each(x.y, y.y), Each(x.z, y.z), Each(x.w, y.w)}; }
    static __device__ __forceinline__ Out Result(const Val &v) { return v; }
};
template <> struct FoldLane<HalfBits, ROP_MAX> : HalfMaxLane<ROP_MAX> {};
template <> struct FoldLane<HalfBits, ROP_MIN> : HalfMaxLane<ROP_MIN> {};

// bf16: the upper element as the fp32 that the whole word is (the lower element hangs on as low mantissa bits, which only
// decide between equal upper elements; an infinity becomes a NaN by them, and is then told as one), the lower one shifted up.
template <int OP> struct Bf16MaxLane {
    typedef SplitVec Val;
    typedef V4 Raw;
    typedef V4 Out;
    typedef VecLane<Bf16Bits, OP> Exact;
    typedef SpecialHalves<0x7f80u, OP> Special;
    static constexpr bool kChecked = true;
    static __device__ __forceinline__ Raw Load(const void *base, uint32_t pos) { return Load16<ACC_VEC16_ANY>(base, pos); }
    static __device__ __forceinline__ Val Value(const Raw &r, const void *) { return Val{r, r << 16}; }
    static __device__ __forceinline__ uint32_t Each(uint32_t x, uint32_t y)
    {
        const float a = __uint_as_float(x), b = __uint_as_float(y);
        return __float_as_uint(OP == ROP_MAX ? __builtin_elementwise_maximum(a, b) : __builtin_elementwise_minimum(a, b));
    }
    static __device__ __forceinline__ V4 Each(V4 x, V4 y) { return V4{Each(x.x, y.x), Each(x.y, y.y), Each(x.z, y.z), Each(x.w, y.w)}; }
    static __device__ __forceinline__ Val Combine(const Val &x, const Val &y) { return Val{Each(x.a, y.a), Each(x.b, y.b)}; }
    static __device__ __forceinline__ uint32_t Join(uint32_t upper, uint32_t lower) { return __builtin_amdgcn_perm(upper, lower, 0x07060302u); }
    static __device__ __forceinline__ Out Result(const Val &v)
    {
        return V4{Join(v.a.x, v.b.x), Join(v.a.y, v.b.y), Join(v.a.z, v.b.z), Join(v.a.w, v.b.w)};
    }
};
template <> struct FoldLane<Bf16Bits, ROP_MAX> : Bf16MaxLane<ROP_MAX> {};
template <> struct FoldLane<Bf16Bits, ROP_MIN> : Bf16MaxLane<ROP_MIN> {};

// Keeps the compiler from moving memory accesses over this point (it sinks loads to their first use otherwise).
__device__ __forceinline__ void PinAccesses() { asm volatile("" ::: "memory"); }

// U values per lane to nbytes at every destination (positions at or behind nbytes are dropped by the buffer range check).
template <uint32_t POLICY, uint32_t U>
__device__ __forceinline__ void StoreEach(void *const *__restrict__ dst, uint32_t ndst, uint64_t off, uint32_t nbytes,
    const uint32_t (&pos)[U], const V4 (&v)[U])
{
    for (uint32_t k = 0; k < ndst; k++) {
        const BufferRsrc r = MakeBuffer(static_cast<char *>(dst[k]) + off, nbytes);
#pragma unroll
        for (uint32_t u = 0; u < U; u++) {
            BufferStore16<POLICY>(r, pos[u], v[u]);
        }
    }
}
template <uint32_t U>
__device__ __forceinline__ void StoreByFlags(const FusedDesc &d, void *const *__restrict__ dst, uint64_t off, uint32_t nbytes,
    const uint32_t (&pos)[U], const V4 (&v)[U])
{
    if (d.flags & kFusedThroughStores) {
        StoreEach<STORE_THROUGH>(dst, d.ndst, off, nbytes, pos, v);
    } else if (d.flags & kFusedOrdinaryStores) {
        StoreEach<STORE_ORDINARY>(dst, d.ndst, off, nbytes, pos, v);
    } else {
        StoreEach<STORE_NT>(dst, d.ndst, off, nbytes, pos, v);
    }
}

// Positions of a lane's vectors in a tile, and where it reads: a lane behind the last vector of a piece that is no whole
// tile reads that one again and drops the result.
template <uint32_t U> __device__ __forceinline__ void TilePositions(uint32_t (&pos)[U])
{
#pragma unroll
    for (uint32_t u = 0; u < U; u++) {
        pos[u] = (u * kBlockThreads + threadIdx.x) * 16u;
    }
}
template <uint32_t U> __device__ __forceinline__ void ReadPositions(const uint32_t (&pos)[U], uint32_t nbytes, uint32_t (&at)[U])
{
#pragma unroll
    for (uint32_t u = 0; u < U; u++) {
        at[u] = pos[u] < nbytes ? pos[u] : nbytes - 16u;
    }
}

// The rest of an item's body behind its whole tiles, and its ends, of which lane i takes the element at byte i.
__device__ __forceinline__ uint64_t RestOffset(const FusedDesc &d) { return d.bytes / kTileBytes * kTileBytes; }
__device__ __forceinline__ uint32_t RestBytes(const FusedDesc &d) { return uint32_t(d.bytes % kTileBytes); }
__device__ __forceinline__ uint32_t EndBytes(const FusedDesc &d) { return uint32_t(d.head) + d.tail; }
__device__ __forceinline__ uint64_t EndOffset(const FusedDesc &d, uint32_t i) { return (i < d.head ? 0 : d.bytes) + i - d.head; }
static_assert(128 + 16 <= kBlockThreads, "a workgroup takes an item's ends at once");

// Walks a launch's tiles with a grid stride: whole(d, ahead(d), off) for each whole tile, rest(d, ends) for each tile behind them.
// A workgroup keeps its item while its tiles stay inside it; the next item, and what `ahead` fetches for it, is looked up
// ahead of the current tile's loads, so that the chain of dependent loads (table, item, pointer) completes behind those.
template <typename Ahead, typename Whole, typename Rest>
__device__ __forceinline__ void WalkTiles(const FusedDesc *__restrict__ items, uint32_t nitems, uint32_t nall, uint32_t nwhole, uint32_t ntiles,
    uint32_t tilesPerItem, Ahead ahead, Whole whole, Rest rest)
{
    uint32_t tile = blockIdx.x;
    if (tile < nwhole) {
        FusedDesc d = items[ItemOfTile(items, nitems, tile, tilesPerItem)];
        uint32_t dEnd = d.tile0 + uint32_t(d.bytes / kTileBytes);
        auto a = ahead(d);
        for (;;) {
            const uint32_t next = tile + gridDim.x;
            FusedDesc dn = d;
            uint32_t dnEnd = dEnd;
            auto an = a;
            if (next < nwhole && next >= dEnd) {
                dn = items[ItemOfTile(items, nitems, next, tilesPerItem)];
                dnEnd = dn.tile0 + uint32_t(dn.bytes / kTileBytes);
                an = ahead(dn);
            }
            whole(d, a, uint64_t(tile - d.tile0) * kTileBytes);
            tile = next;
            if (tile >= nwhole) {
                break;
            }
            d = dn;
            dEnd = dnEnd;
            a = an;
        }
    }
    for (; tile < ntiles; tile += gridDim.x) {
        const uint32_t r = tile - nwhole;
        const bool ends = r >= nall;
        const FusedDesc d = items[ends ? r - nall : r];
        rest(d, ends);
    }
}

// ---- fused chain: read every source once, combine in schedule order, write every destination ----------
// Sources go in straight-line code, all loads of a step in front of its combines: a guard per source makes the compiler wait
// for the loads issued so far at every guard, and a lane then has 8 loads in flight instead of 32.
template <typename L, uint32_t N, uint32_t U>
__device__ __forceinline__ void ChainLoad(const void *const *__restrict__ src, uint64_t off, const uint32_t (&at)[U], typename L::Raw (&v)[N][U])
{
#pragma unroll
    for (uint32_t j = 0; j < N; j++) {
        const char *s = static_cast<const char *>(src[j]) + off;
#pragma unroll
        for (uint32_t u = 0; u < U; u++) {
            v[j][u] = L::Load(s, at[u]);
        }
    }
    PinAccesses();
}
// Folds N sources into acc; FIRST: the first of them starts it.
template <typename L, typename T, int OP, uint32_t N, uint32_t U, bool FIRST>
__device__ __forceinline__ void ChainFold(const void *const *__restrict__ src, const typename L::Raw (&v)[N][U], uint64_t accLeft, typename L::Val (&acc)[U])
{
#pragma unroll
    for (uint32_t j = 0; j < N; j++) {
        if (FIRST && j == 0) {
#pragma unroll
            for (uint32_t u = 0; u < U; u++) {
                acc[u] = L::Value(v[0][u], src[0]);
            }
        } else if (OrderMatters<T, OP>::value && !L::kChecked && ((accLeft >> j) & 1ull)) {
            // the flag is the same for the whole wave: a branch, not both results and a select per element
#pragma unroll
            for (uint32_t u = 0; u < U; u++) {
                acc[u] = L::Combine(acc[u], L::Value(v[j][u], src[j]));
            }
        } else {
#pragma unroll
            for (uint32_t u = 0; u < U; u++) {
                acc[u] = L::Combine(L::Value(v[j][u], src[j]), acc[u]);
            }
        }
    }
}
template <typename L, typename T, int OP, uint32_t N, uint32_t U, bool FIRST>
__device__ __forceinline__ void ChainBatch(const void *const *__restrict__ src, uint64_t off, const uint32_t (&at)[U], uint64_t accLeft,
    typename L::Val (&acc)[U])
{
    typename L::Raw v[N][U];
    ChainLoad<L, N, U>(src, off, at, v);
    ChainFold<L, T, OP, N, U, FIRST>(src, v, accLeft, acc);
}

// Makes what comes after it wait for these values.
template <uint32_t U> __device__ __forceinline__ void HoldBack(SplitVec (&x)[U])
{
#pragma unroll
    for (uint32_t u = 0; u < U; u++) {
        asm volatile("" : "+v"(x[u].a), "+v"(x[u].b)::"memory");
    }
}
template <uint32_t U> __device__ __forceinline__ void HoldBack(V4 (&x)[U])
{
#pragma unroll
    for (uint32_t u = 0; u < U; u++) {
        asm volatile("" : "+v"(x[u])::"memory");
    }
}

template <typename L, uint32_t U> __device__ __forceinline__ void ChainResult(const typename L::Val (&acc)[U], typename L::Out (&x)[U])
{
#pragma unroll
    for (uint32_t u = 0; u < U; u++) {
        x[u] = L::Result(acc[u]);
    }
}
template <typename L, typename T, int OP, uint32_t N, uint32_t U>
__device__ __forceinline__ void ChainWhole(const void *const *__restrict__ src, uint64_t off, const uint32_t (&at)[U], uint64_t accLeft,
    typename L::Out (&x)[U])
{
    typename L::Raw v[N][U];
    typename L::Val acc[U];
    ChainLoad<L, N, U>(src, off, at, v);
    if constexpr (L::kChecked && N > 1) {
        // Each question is asked of a wave.  A first vector that holds a NaN or zeros of both signs: by the rule at once.
        typename L::Special first;
        first.SeeNan(v[0][0]);
        first.SeePlus(v[0][0]);
        first.SeeMinus(v[0][0]);
        bool byRule = __any(first.Nan()) || (__any(first.Plus()) && __any(first.Minus()));
        if (!byRule) {
            ChainFold<L, T, OP, N, U, true>(src, v, accLeft, acc);
            ChainResult<L, U>(acc, x);
            typename L::Special any;
#pragma unroll
            for (uint32_t u = 0; u < U; u++) {
                any.SeeAny(x[u]);
            }
            if (__builtin_expect(__any(any.Any()), 0)) {
                typename L::Special result;
#pragma unroll
                for (uint32_t u = 0; u < U; u++) {
                    result.SeeNan(x[u]);
                    result.SeeTaken(x[u]);
                }
                byRule = __any(result.Nan());
                if (!byRule && __any(result.Taken())) {
                    typename L::Special sources;
#pragma unroll
                    for (uint32_t j = 0; j < N; j++) {
#pragma unroll
                        for (uint32_t u = 0; u < U; u++) {
                            sources.SeePassed(v[j][u]);
                        }
                    }
                    byRule = __any(sources.Passed());
                }
            }
        }
        if (__builtin_expect(byRule, 0)) {
            ChainFold<typename L::Exact, T, OP, N, U, true>(src, v, accLeft, x);
        }
    } else {
        ChainFold<L, T, OP, N, U, true>(src, v, accLeft, acc);
        ChainResult<L, U>(acc, x);
    }
}

// The chain's value at U positions of a lane, `off` behind the item's pointers: up to 8 sources, all in flight together (src is
// only indexed with constants: a caller may keep the pointers in registers).
template <typename L, typename T, int OP, uint32_t U>
__device__ __forceinline__ void ChainFew(uint32_t nsrc, uint64_t accLeft, const void *const *__restrict__ src, uint64_t off, const uint32_t (&at)[U],
    typename L::Out (&x)[U])
{
    switch (nsrc) {
        case 1: ChainWhole<L, T, OP, 1, U>(src, off, at, accLeft, x); break;
        case 2: ChainWhole<L, T, OP, 2, U>(src, off, at, accLeft, x); break;
        case 3: ChainWhole<L, T, OP, 3, U>(src, off, at, accLeft, x); break;
        case 4: ChainWhole<L, T, OP, 4, U>(src, off, at, accLeft, x); break;
        case 5: ChainWhole<L, T, OP, 5, U>(src, off, at, accLeft, x); break;
        case 6: ChainWhole<L, T, OP, 6, U>(src, off, at, accLeft, x); break;
        case 7: ChainWhole<L, T, OP, 7, U>(src, off, at, accLeft, x); break;
        default: ChainWhole<L, T, OP, 8, U>(src, off, at, accLeft, x); break;
    }
}
// More than 8 sources: two sets of 4, one in flight while the other is folded.
template <typename L, typename T, int OP, uint32_t U>
__device__ __forceinline__ void ChainMany(uint32_t nsrc, uint64_t accLeft, const void *const *__restrict__ src, uint64_t off, const uint32_t (&at)[U],
    typename L::Out (&x)[U])
{
    constexpr uint32_t N = 4;
    typename L::Val acc[U];
    typename L::Raw va[N][U], vb[N][U];
    ChainLoad<L, N, U>(src, off, at, va);
    ChainLoad<L, N, U>(src + N, off, at, vb);
    ChainFold<L, T, OP, N, U, true>(src, va, accLeft, acc);
    uint32_t j = N;               // vb holds sources j ... j + N - 1
#pragma nounroll
    for (; j + 3 * N <= nsrc; j += 2 * N) {
        ChainLoad<L, N, U>(src + j + N, off, at, va);
        ChainFold<L, T, OP, N, U, false>(src + j, vb, accLeft >> j, acc);
        ChainLoad<L, N, U>(src + j + 2 * N, off, at, vb);
        ChainFold<L, T, OP, N, U, false>(src + j + N, va, accLeft >> (j + N), acc);
    }
    if (j + 2 * N <= nsrc) {
        ChainLoad<L, N, U>(src + j + N, off, at, va);
        ChainFold<L, T, OP, N, U, false>(src + j, vb, accLeft >> j, acc);
        ChainFold<L, T, OP, N, U, false>(src + j + N, va, accLeft >> (j + N), acc);
        j += 2 * N;
    } else {
        ChainFold<L, T, OP, N, U, false>(src + j, vb, accLeft >> j, acc);
        j += N;
    }
    switch (nsrc - j) {
        case 1: ChainBatch<L, T, OP, 1, U, false>(src + j, off, at, accLeft >> j, acc); break;
        case 2: ChainBatch<L, T, OP, 2, U, false>(src + j, off, at, accLeft >> j, acc); break;
        case 3: ChainBatch<L, T, OP, 3, U, false>(src + j, off, at, accLeft >> j, acc); break;
        default: break;
    }
    ChainResult<L, U>(acc, x);
}
template <typename L, typename T, int OP, uint32_t U>
__device__ __forceinline__ void ChainValue(const FusedDesc &d, const void *const *__restrict__ src, uint64_t off, const uint32_t (&at)[U],
    typename L::Out (&x)[U])
{
    if (d.nsrc <= 8) {
        ChainFew<L, T, OP, U>(d.nsrc, d.accLeftMask, src, off, at, x);
    } else {
        ChainMany<typename L::Exact, T, OP, U>(d.nsrc, d.accLeftMask, src, off, at, x);
    }
}
// The same with two sources in flight at a time: a source is requested when the one two before it is folded.
template <typename L, typename T, int OP, uint32_t U>
__device__ __forceinline__ void ChainSlow(const FusedDesc &d, const void *const *__restrict__ src, uint64_t off, const uint32_t (&at)[U],
    typename L::Out (&x)[U])
{
    const uint32_t nsrc = d.nsrc;
    const uint64_t accLeft = d.accLeftMask;
    typename L::Val acc[U];
    if (nsrc == 1) {
        ChainBatch<L, T, OP, 1, U, true>(src, off, at, accLeft, acc);
        ChainResult<L, U>(acc, x);
        return;
    }
    typename L::Raw va[1][U], vb[1][U];
    ChainLoad<L, 1, U>(src, off, at, va);
    ChainLoad<L, 1, U>(src + 1, off, at, vb);
    ChainFold<L, T, OP, 1, U, true>(src, va, accLeft, acc);
    HoldBack(acc);
    uint32_t j = 1;               // vb holds source j
#pragma nounroll
    for (; j + 3 <= nsrc; j += 2) {
        ChainLoad<L, 1, U>(src + j + 1, off, at, va);
        ChainFold<L, T, OP, 1, U, false>(src + j, vb, accLeft >> j, acc);
        HoldBack(acc);
        ChainLoad<L, 1, U>(src + j + 2, off, at, vb);
        ChainFold<L, T, OP, 1, U, false>(src + j + 1, va, accLeft >> (j + 1), acc);
        HoldBack(acc);
    }
    if (j + 2 <= nsrc) {
        ChainLoad<L, 1, U>(src + j + 1, off, at, va);
        ChainFold<L, T, OP, 1, U, false>(src + j, vb, accLeft >> j, acc);
        ChainFold<L, T, OP, 1, U, false>(src + j + 1, va, accLeft >> (j + 1), acc);
    } else {
        ChainFold<L, T, OP, 1, U, false>(src + j, vb, accLeft >> j, acc);
    }
    ChainResult<L, U>(acc, x);
}

// U vectors per lane of a tile, or of a piece of `nbytes` (a multiple of 16).
template <typename T, int OP, bool WHOLE, bool SLOW, uint32_t U>
__device__ __forceinline__ void ChainTile(const FusedDesc &d, const void *const *__restrict__ src, void *const *__restrict__ dst, uint64_t off, uint32_t nbytes)
{
    typedef FoldLane<T, OP> Vec;
    typedef WordLane<T, OP> Words;
    uint32_t pos[U], at[U];
    V4 acc[U];
    TilePositions(pos);
    ReadPositions(pos, WHOLE ? kTileBytes : nbytes, at);
    if (sizeof(T) == 1 && (d.flags & kFusedWordSources)) {
        ChainSlow<Words, T, OP, U>(d, src, off, at, acc);     // (all in flight takes more registers than there are)
    } else if (SLOW) {
        ChainSlow<typename Vec::Exact, T, OP, U>(d, src, off, at, acc);
    } else {
        ChainValue<Vec, T, OP, U>(d, src, off, at, acc);
    }
    StoreByFlags(d, dst, off, WHOLE ? kTileBytes : nbytes, pos, acc);
}

// An item's rest, or its ends.
template <typename T, int OP, bool SLOW = false>
__device__ __forceinline__ void ChainRest(const FusedDesc &d, bool ends, const void *const *__restrict__ src, void *const *__restrict__ dst)
{
    if (!ends) {
        const uint64_t off = RestOffset(d);
        const uint32_t n = RestBytes(d);
        if (n == 0) {
            return;
        }
        if (n <= kBlockThreads * 16u) {
            ChainTile<T, OP, false, false, 1>(d, src, dst, off, n);
        } else {
            ChainTile<T, OP, false, SLOW, kChainVec>(d, src, dst, off, n);
        }
    } else {
        const uint32_t i = threadIdx.x * uint32_t(sizeof(T));
        if (i < EndBytes(d)) {
            const uint64_t off = EndOffset(d, i);
            const uint32_t at[1] = {0};
            T acc[1];
            ChainValue<ElemLane<T, OP>, T, OP, 1>(d, src, off, at, acc);
            for (uint32_t k = 0; k < d.ndst; k++) {
                StoreElem<T>(dst[k], off, acc[0]);
            }
        }
    }
}

// Two forms.  Measured, us, this kernel's loads guarded one by one (before) / all in flight / two sources in flight: all-reduce, 8
// ranks, fp32, 2 MiB per rank 7.3 / 7.3 / 7.5, 6 MiB 20.1 / 17.5 / 18.9, 8 MiB 23.9 / 22.2 / 23.9; reduce-scatter, 8 ranks, fp32, blocks of 8 MiB
// 97.0 / 101.0 / 98.6, 16 MiB 192.7 / 200.1 / 190.8; 16 ranks, bf16 maximum, 512 KiB 27.6 / 25.4 / 23.7, 16 MiB 777 / 767 / 755.
// SLOW = false has all loads of a tile in flight, the shortest way through a tile, for launches of a tile per CU or fewer.
// SLOW = true has two sources' in flight and 70 registers instead of 161 (fp32, fp16 sum; bf16 120 instead of 254, int8 102 - 115
// instead of 253 - 256): where tiles follow one another, and for many sources into one destination, workgroups that ask for
// less at a time move more.
template <typename T, int OP, bool SLOW>
__global__ void __launch_bounds__(kBlockThreads, 2) ChainKernel(const FusedDesc *__restrict__ items, uint32_t nitems, uint32_t nall, uint32_t nwhole,
    uint32_t ntiles, const void *const *__restrict__ srcPool, void *const *__restrict__ dstPool, uint32_t tilesPerItem)
{
    WalkTiles(items, nitems, nall, nwhole, ntiles, tilesPerItem, [](const FusedDesc &) { return 0; },
        [&](const FusedDesc &d, int, uint64_t off) { ChainTile<T, OP, true, SLOW, kChainVec>(d, srcPool + d.srcBase, dstPool + d.dstBase, off, kTileBytes); },
        [&](const FusedDesc &d, bool ends) { ChainRest<T, OP, SLOW>(d, ends, srcPool + d.srcBase, dstPool + d.dstBase); });
}

// ---- pure data movement: one source, m destinations ------------------------------------------------------
// The chain kernel's copy path with nothing else in the kernel: about 40 registers instead of 170+, so eight
// workgroups fit on a CU where the chain kernel fits two.  A copy keeps only 4 loads per lane in flight, and its
// rate comes from how many waves do that at once (measured, 1 GiB copy: 5.1 TB/s through the chain kernel,
// 6.3 TB/s for a plain copy kernel at full occupancy).
typedef VecLane<uint8_t, ROP_SUM> MoveLane;

template <bool WHOLE>
__device__ __forceinline__ void CopyTile(const FusedDesc &d, const void *s, void *const *__restrict__ dst, uint64_t off, uint32_t nbytes)
{
    uint32_t pos[kChainVec], at[kChainVec];
    V4 v[1][kChainVec];
    TilePositions(pos);
    ReadPositions(pos, WHOLE ? kTileBytes : nbytes, at);
    ChainLoad<MoveLane, 1, kChainVec>(&s, off, at, v);
    // All loads here, on every way to the stores: without it the compiler, which cannot tell on which way they were waited for,
    // makes the next tile's loads wait for this tile's stores (uniform all-to-all, us, with that wait / without: 8 ranks 32 MiB 86.8 / 84.7,
    // 256 MiB 708 / 688; 16 ranks 256 MiB 1445 / 1402).
    HoldBack(v[0]);
    StoreByFlags(d, dst, off, WHOLE ? kTileBytes : nbytes, pos, v[0]);
}
__device__ __forceinline__ void CopyRest(const FusedDesc &d, bool ends, const void *s, void *const *__restrict__ dst)
{
    if (!ends) {
        if (RestBytes(d) != 0) {
            CopyTile<false>(d, s, dst, RestOffset(d), RestBytes(d));
        }
    } else if (threadIdx.x < EndBytes(d)) {
        const uint64_t off = EndOffset(d, threadIdx.x);
        const uint8_t b = LoadElem<uint8_t>(s, off);
        for (uint32_t k = 0; k < d.ndst; k++) {
            StoreElem<uint8_t>(dst[k], off, b);
        }
    }
}

// Same arguments and tables as the chain kernel; every item has exactly one source.  (A template only so that the
// definition may sit in this header; Variant is unused.)
template <int Variant>
__global__ void __launch_bounds__(kBlockThreads) CopyKernel(const FusedDesc *__restrict__ items, uint32_t nitems, uint32_t nall, uint32_t nwhole,
    uint32_t ntiles, const void *const *__restrict__ srcPool, void *const *__restrict__ dstPool, uint32_t tilesPerItem)
{
    WalkTiles(items, nitems, nall, nwhole, ntiles, tilesPerItem, [&](const FusedDesc &d) { return srcPool[d.srcBase]; },
        [&](const FusedDesc &d, const void *s, uint64_t off) { CopyTile<true>(d, s, dstPool + d.dstBase, off, kTileBytes); },
        [&](const FusedDesc &d, bool ends) { CopyRest(d, ends, srcPool[d.srcBase], dstPool + d.dstBase); });
}

// ---- small-segment gather: LDS staging ---------------------------------------------------------------------
// An all-to-all-v of many short segments (a few hundred bytes each, at any byte offset in the send and receive
// buffers) is all overhead in the tile kernels: a descriptor search per tile, a head / body / tail split per
// segment, unaligned accesses.  Here a wave takes a whole segment: it reads the aligned 16-byte granules that cover
// the source bytes into its share of LDS (coalesced, aligned loads; the bytes in front of and behind the segment that
// come along lie in the same granules as valid bytes), then every lane picks the 16 bytes of one aligned granule of
// the destination out of LDS at whatever offset they sit and stores them aligned; the two ragged ends go byte by
// byte.  Segments are dealt to waves round robin, no search.
// Stands where the reference's AIV kernel stages small all-to-all-v slices through its unified buffer
// (ALG/base/alg_aiv_template/aiv_all_to_all_v_910b.h:39-222); nothing of it is reused.
constexpr uint32_t kGatherLdsPerWave = kGatherMaxBytes + 32;

template <int Variant>
__global__ void __launch_bounds__(kBlockThreads) GatherKernel(const SegDesc *__restrict__ segs, uint32_t nsegs)
{
    __shared__ __attribute__((aligned(16))) uint8_t lds[(kBlockThreads / 64) * kGatherLdsPerWave];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    uint8_t *mine = lds + wave * kGatherLdsPerWave;
    const uint32_t wavesPerBlock = kBlockThreads / 64;
    for (uint32_t i = blockIdx.x * wavesPerBlock + wave; i < nsegs; i += gridDim.x * wavesPerBlock) {
        const SegDesc d = segs[i];
        const uint32_t n = uint32_t(d.bytes);
        if (n == 0) {
            continue;
        }
        const uintptr_t s = reinterpret_cast<uintptr_t>(d.src), t = reinterpret_cast<uintptr_t>(d.dst);
        const uintptr_t s0 = s & ~uintptr_t(15);
        const uint32_t delta = uint32_t(s - s0);                       // where the segment starts inside LDS
        const uint32_t nin = (delta + n + 15u) >> 4;                   // granules to read
        for (uint32_t v = lane; v < nin; v += 64) {
            const V4 x = __builtin_nontemporal_load((const GlobalV4 *)(s0 + uintptr_t(v) * 16));
            *(LdsV4 *)(mine + v * 16) = x;
        }
        // LDS operations of one wave complete in order; the compiler must keep that order too
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const uintptr_t t0 = (t + 15) & ~uintptr_t(15);               // first aligned granule inside the destination
        const uint32_t head = uint32_t(t0 - t) < n ? uint32_t(t0 - t) : n;
        const uint32_t body = (n - head) >> 4;                         // whole granules
        const uint32_t tail = n - head - body * 16;
        for (uint32_t v = lane; v < body; v += 64) {
            const LdsV4U *from = (const LdsV4U *)(mine + delta + head + v * 16);
            const V4U x = *from;
            __builtin_nontemporal_store(V4{x.x, x.y, x.z, x.w}, (GlobalV4 *)(t0 + uintptr_t(v) * 16));
        }
        if (lane < head) {
            StoreElem<uint8_t>(d.dst, lane, mine[delta + lane]);
        }
        if (lane < tail) {
            const uint32_t at = head + body * 16 + lane;
            StoreElem<uint8_t>(d.dst, at, mine[delta + at]);
        }
        // the next segment's loads into LDS must not overtake this segment's reads
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
}

// ---- fused perfect tree (halving-doubling): leaves pairwise bottom-up ----------------------------------
// v[i] = v[i] (+) v[i+w] for w = 1, 2, 4, ...  Same association as the flat loop, evaluated in groups of 8 leaves: a
// group's leaves come in two sets of 4, and while one set is folded the other one's loads, then the next group's, are in
// flight; the group results go through a binary counter.
constexpr uint32_t kTreeGroup = 8;

// N leaves from leaf 0 of `src` on (two pool entries each, the second one of a folded rank pair or null).
template <typename L, uint32_t N, uint32_t U>
__device__ __forceinline__ void TreeLoad(const void *const *__restrict__ src, uint64_t off, const uint32_t (&at)[U], typename L::Val (&v)[N][U])
{
#pragma unroll
    for (uint32_t i = 0; i < N; i++) {
        const char *s = static_cast<const char *>(src[2 * i]) + off;
#pragma unroll
        for (uint32_t u = 0; u < U; u++) {
            v[i][u] = L::Load(s, at[u]);
        }
    }
    PinAccesses();
}
// The second sources of the leaves that have one: together where all of them do, the usual case.
template <typename L, uint32_t N, uint32_t U>
__device__ __forceinline__ void TreePairs(const void *const *__restrict__ src, uint64_t off, const uint32_t (&at)[U], typename L::Val (&v)[N][U])
{
    bool all = true;
#pragma unroll
    for (uint32_t i = 0; i < N; i++) {
        all = all && src[2 * i + 1] != nullptr;
    }
    if (all) {
        typename L::Val w[N][U];
        TreeLoad<L, N, U>(src + 1, off, at, w);
#pragma unroll
        for (uint32_t i = 0; i < N; i++) {
#pragma unroll
            for (uint32_t u = 0; u < U; u++) {
                v[i][u] = L::Combine(v[i][u], w[i][u]);
            }
        }
    } else {
#pragma unroll
        for (uint32_t i = 0; i < N; i++) {
            if (src[2 * i + 1] != nullptr) {
                typename L::Val w[1][U];
                TreeLoad<L, 1, U>(src + 2 * i + 1, off, at, w);
#pragma unroll
                for (uint32_t u = 0; u < U; u++) {
                    v[i][u] = L::Combine(v[i][u], w[0][u]);
                }
            }
        }
    }
}
// N leaves pairwise into x.  8-bit sums: the compiler keeps them apart as even and odd bytes from one level to the next and past the
// set's end, which takes 312 registers in the plain kernel and leaves a CU one workgroup; put together at a set's end it takes 223,
// and two fit.  Halving-doubling reduce-scatter, 8 ranks, us, 8 leaves in one set (before) / kept apart / put together: blocks of 1 MiB
// 12.2 / 12.9 / 10.8, 2 MiB 23.7 / 26.1 / 21.5, 8 MiB 101.5 / 99.5 / 99.8; all-reduce 8 ranks 8 MiB 24.7 / 20.8 / 21.3; reduce 16 ranks 64 MiB
// 193 / 182 / 189.  (Other types take 253 to 292 and lose by it: all-reduce 16 ranks fp32 4 MiB 19.6 / 20.2, int64 19.7 / 20.2.)
template <typename L, uint32_t N, uint32_t U>
__device__ __forceinline__ void TreeFold(typename L::Val (&v)[N][U], typename L::Val (&x)[U])
{
#pragma unroll
    for (uint32_t w = 1; w < N; w <<= 1) {
#pragma unroll
        for (uint32_t i = 0; i + w < N; i += 2 * w) {
#pragma unroll
            for (uint32_t u = 0; u < U; u++) {
                v[i][u] = L::Combine(v[i][u], v[i + w][u]);
            }
        }
    }
#pragma unroll
    for (uint32_t u = 0; u < U; u++) {
        x[u] = v[0][u];
    }
    if constexpr (L::kHoldBack) {
        HoldBack(x);
    }
}
template <typename L, uint32_t U>
__device__ __forceinline__ void TreeJoin(const typename L::Val (&a)[U], typename L::Val (&x)[U])
{
#pragma unroll
    for (uint32_t u = 0; u < U; u++) {
        x[u] = L::Combine(a[u], x[u]);
    }
}
template <typename L, uint32_t N, uint32_t U>
__device__ __forceinline__ void TreeSet(const void *const *__restrict__ src, uint64_t off, const uint32_t (&at)[U], typename L::Val (&x)[U])
{
    typename L::Val v[N][U];
    TreeLoad<L, N, U>(src, off, at, v);
    TreePairs<L, N, U>(src, off, at, v);
    TreeFold<L, N, U>(v, x);
}

// The tree's value at U positions of a lane, `off` behind the item's pointers.
template <typename L, uint32_t U>
__device__ __forceinline__ void TreeValue(const FusedDesc &d, const void *const *__restrict__ src, uint64_t off, const uint32_t (&at)[U],
    typename L::Val (&x)[U])
{
    if (d.nleaf < kTreeGroup) {
        if (d.nleaf == 4) {
            TreeSet<L, 4, U>(src, off, at, x);
        } else if (d.nleaf == 2) {
            TreeSet<L, 2, U>(src, off, at, x);
        } else {
            TreeSet<L, 1, U>(src, off, at, x);
        }
        return;
    }
    const uint32_t ngroups = d.nleaf / kTreeGroup;   // 1, 2 or 4
    typename L::Val l0[U], l1[U], y[U];              // pending left operands of the upper levels
    auto count = [&](uint32_t gi) {
        if ((gi & 1u) == 0) {
#pragma unroll
            for (uint32_t u = 0; u < U; u++) {
                l0[u] = x[u];
            }
        } else {
            TreeJoin<L, U>(l0, x);
            if ((gi & 2u) == 0) {
#pragma unroll
                for (uint32_t u = 0; u < U; u++) {
                    l1[u] = x[u];
                }
            } else {
                TreeJoin<L, U>(l1, x);
            }
        }
    };
    if (d.flags & kFusedPairs) {
#pragma nounroll
        for (uint32_t gi = 0; gi < ngroups; gi++) {
            const void *const *gs = src + 2 * gi * kTreeGroup;
            TreeSet<L, 4, U>(gs, off, at, y);
            TreeSet<L, 4, U>(gs + 8, off, at, x);
            TreeJoin<L, U>(y, x);
            count(gi);
        }
        return;
    }
    typename L::Val va[4][U], vb[4][U];
    TreeLoad<L, 4, U>(src, off, at, va);
    TreeLoad<L, 4, U>(src + 8, off, at, vb);
    uint32_t gi = 0;
#pragma nounroll
    for (; gi + 1 < ngroups; gi++) {
        const void *const *next = src + 2 * (gi + 1) * kTreeGroup;
        TreeFold<L, 4, U>(va, y);
        TreeLoad<L, 4, U>(next, off, at, va);
        TreeFold<L, 4, U>(vb, x);
        TreeLoad<L, 4, U>(next + 8, off, at, vb);
        TreeJoin<L, U>(y, x);
        count(gi);
    }
    TreeFold<L, 4, U>(va, y);
    TreeFold<L, 4, U>(vb, x);
    TreeJoin<L, U>(y, x);
    count(gi);
}

template <typename T, int OP>
__device__ __forceinline__ void TreeRest(const FusedDesc &d, bool ends, const void *const *__restrict__ src, void *const *__restrict__ dst)
{
    if (!ends) {
        const uint64_t off = RestOffset(d);
        const uint32_t n = RestBytes(d);
        if (n == 0) {
            return;
        }
        uint32_t pos[kChainVec], at[kChainVec];
        V4 x[kChainVec];
        TilePositions(pos);
        ReadPositions(pos, n, at);
        TreeValue<VecLane<T, OP>, kChainVec>(d, src, off, at, x);
        StoreByFlags(d, dst, off, n, pos, x);
    } else {
        const uint32_t i = threadIdx.x * uint32_t(sizeof(T));
        if (i < EndBytes(d)) {
            const uint64_t off = EndOffset(d, i);
            const uint32_t at[1] = {0};
            T x[1];
            TreeValue<ElemLane<T, OP>, 1>(d, src, off, at, x);
            for (uint32_t k = 0; k < d.ndst; k++) {
                StoreElem<T>(dst[k], off, x[0]);
            }
        }
    }
}

template <typename T, int OP>
__global__ void __launch_bounds__(kBlockThreads) TreeKernel(const FusedDesc *__restrict__ items, uint32_t nitems, uint32_t nall, uint32_t nwhole,
    uint32_t ntiles, const void *const *__restrict__ srcPool, void *const *__restrict__ dstPool, uint32_t tilesPerItem)
{
    uint32_t pos[kChainVec];
    TilePositions(pos);
    WalkTiles(items, nitems, nall, nwhole, ntiles, tilesPerItem, [](const FusedDesc &) { return 0; },
        [&](const FusedDesc &d, int, uint64_t off) {
            V4 x[kChainVec];
            TreeValue<VecLane<T, OP>, kChainVec>(d, srcPool + d.srcBase, off, pos, x);
            StoreByFlags(d, dstPool + d.dstBase, off, kTileBytes, pos, x);
        },
        [&](const FusedDesc &d, bool ends) { TreeRest<T, OP>(d, ends, srcPool + d.srcBase, dstPool + d.dstBase); });
}

// ---- fused general expression: a stack machine over registers -----------------------------------------
// Handles what is neither a chain nor a perfect tree (a ring or halving-doubling schedule whose
// operands are themselves mesh chains, for one).  The item's sources come in evaluation order; after
// source j the two topmost values are folded ops[j] & 7 times, bit 8 + i saying which of the two is
// the left operand in fold i.  The op words of a launch follow its item table in memory.
// The stack lives in registers: its depth is a wave-uniform number, so every access goes through a
// switch with constant indices.  Sources are loaded in batches like the chain kernel's.
// Two shapes: expressions that need at most 4 values (a chain of chains, a 4-leaf tree of chains) run
// with 4 vectors per lane like the chain kernel, deeper ones (up to 8 values) with 2.
constexpr uint32_t kStackVecDeep = 2;
constexpr uint32_t kStackShallowDepth = 4;
constexpr uint32_t kStackTeamBatch = 8;
// The plain kernel issues the loads of 4 sources together: with 8 it needs every register a wave can have, one
// workgroup fits a CU and nothing hides the table look-ups between its tiles (two-level reduce-scatter of 8 x 256 MiB
// 426 -> 417 us, reduce 434 -> 415 us, all-reduce of 8 x 16 MiB 52 -> 47 us).  The team form, one workgroup per CU by
// its LDS, keeps 8.
constexpr uint32_t kStackPlainBatch = 4;

template <typename V, uint32_t U> struct StackVal {
    V x[U];
};

// The values below the top one are separate variables, not an array or a struct: a switch over
// parts of one object is merged by the compiler into a single access at a computed offset, which
// moves the object to private memory.  DEEP is a compile-time constant of the enclosing function;
// without it only b0..b2 are ever touched and the others cost no registers.
#define HCCL_STACK_PUT(i, v)              \
    if (DEEP) {                           \
        switch (i) {                      \
            case 0: b0 = (v); break;      \
            case 1: b1 = (v); break;      \
            case 2: b2 = (v); break;      \
            case 3: b3 = (v); break;      \
            case 4: b4 = (v); break;      \
            case 5: b5 = (v); break;      \
            default: b6 = (v); break;     \
        }                                 \
    } else {                              \
        switch (i) {                      \
            case 0: b0 = (v); break;      \
            case 1: b1 = (v); break;      \
            default: b2 = (v); break;     \
        }                                 \
    }
#define HCCL_STACK_GET(i, v)              \
    if (DEEP) {                           \
        switch (i) {                      \
            case 0: (v) = b0; break;      \
            case 1: (v) = b1; break;      \
            case 2: (v) = b2; break;      \
            case 3: (v) = b3; break;      \
            case 4: (v) = b4; break;      \
            case 5: (v) = b5; break;      \
            default: (v) = b6; break;     \
        }                                 \
    } else {                              \
        switch (i) {                      \
            case 0: (v) = b0; break;      \
            case 1: (v) = b1; break;      \
            default: (v) = b2; break;     \
        }                                 \
    }

// Pushes v and folds as its op word says.  A macro: in a function the compiler merges the cases of the switches into one
// access through a pointer.
#define HCCL_STACK_PUSH(v, opword)                                                          \
    {                                                                                       \
        const uint32_t op = (opword);                                                       \
        if (depth > 0) {                                                                    \
            HCCL_STACK_PUT(depth - 1, top)                                                  \
        }                                                                                   \
        top = (v);                                                                          \
        depth++;                                                                            \
        const uint32_t nfold = op & 7u;                                                     \
        _Pragma("nounroll") for (uint32_t f = 0; f < nfold && depth >= 2; f++)              \
        {                                                                                   \
            StackVal<typename L::Val, U> under;                                             \
            HCCL_STACK_GET(depth - 2, under)                                                \
            if (!OrderMatters<T, OP>::value || ((op >> (8 + f)) & 1u)) { /* one for the whole wave */ \
                _Pragma("unroll") for (uint32_t u = 0; u < U; u++)                          \
                {                                                                           \
                    top.x[u] = L::Combine(under.x[u], top.x[u]);                            \
                }                                                                           \
            } else {                                                                        \
                _Pragma("unroll") for (uint32_t u = 0; u < U; u++)                          \
                {                                                                           \
                    top.x[u] = L::Combine(top.x[u], under.x[u]);                            \
                }                                                                           \
            }                                                                               \
            depth--;                                                                        \
        }                                                                                   \
    }

// The expression's value at U positions of a lane, `off` behind the item's pointers.  BATCH sources are loaded together; the
// last batch loads its last source again where it has fewer.
template <typename L, typename T, int OP, uint32_t U, bool DEEP, uint32_t BATCH>
__device__ __forceinline__ void StackValue(const FusedDesc &d, const void *const *__restrict__ src, const uint32_t *__restrict__ ops, uint64_t off,
    const uint32_t (&at)[U], typename L::Val (&x)[U])
{
    StackVal<typename L::Val, U> top;
#pragma unroll
    for (uint32_t u = 0; u < U; u++) {
        top.x[u] = typename L::Val();
    }
    StackVal<typename L::Val, U> b0 = top, b1 = top, b2 = top, b3 = top, b4 = top, b5 = top, b6 = top;
    uint32_t depth = 0;
    const uint32_t nsrc = d.nsrc;
#pragma nounroll
    for (uint32_t j = 0; j < nsrc; j += BATCH) {
        StackVal<typename L::Val, U> v[BATCH];
#pragma unroll
        for (uint32_t jj = 0; jj < BATCH; jj++) {
            const char *s = static_cast<const char *>(src[j + jj < nsrc ? j + jj : nsrc - 1]) + off;
#pragma unroll
            for (uint32_t u = 0; u < U; u++) {
                v[jj].x[u] = L::Load(s, at[u]);
            }
        }
        PinAccesses();
#pragma unroll
        for (uint32_t jj = 0; jj < BATCH; jj++) {
            if (j + jj < nsrc) {
                HCCL_STACK_PUSH(v[jj], ops[j + jj])
            }
        }
    }
#pragma unroll
    for (uint32_t u = 0; u < U; u++) {
        x[u] = top.x[u];
    }
}

// The values of a tile, or of a piece read at `at`, in passes as wide as the depth allows: sink(u, first vector's index, values).
template <typename T, int OP, uint32_t BATCH, typename Sink>
__device__ __forceinline__ void StackTile(const FusedDesc &d, const void *const *__restrict__ src, const uint32_t *__restrict__ ops, uint64_t off,
    const uint32_t (&at)[kChainVec], Sink sink)
{
    typedef VecLane<T, OP> L;
    V4 x[kChainVec];
    if (d.nleaf <= kStackShallowDepth) {      // d.nleaf: the stack depth the item needs
        StackValue<L, T, OP, kChainVec, false, BATCH>(d, src, ops, off, at, x);
        sink(0u, x);
    } else {
#pragma nounroll
        for (uint32_t h = 0; h < kChainVec; h += kStackVecDeep) {
            const uint32_t part[kStackVecDeep] = {h == 0 ? at[0] : at[2], h == 0 ? at[1] : at[3]};
            V4 y[kStackVecDeep];
            StackValue<L, T, OP, kStackVecDeep, true, BATCH>(d, src, ops, off, part, y);
            sink(h, y);
        }
    }
}
static_assert(kChainVec == 4 && kStackVecDeep == 2, "StackTile takes a tile in one pass or in two");

template <typename T, int OP, uint32_t BATCH>
__device__ __forceinline__ void StackStore(const FusedDesc &d, const void *const *__restrict__ src, const uint32_t *__restrict__ ops,
    void *const *__restrict__ dst, uint64_t off, uint32_t nbytes, const uint32_t (&pos)[kChainVec], const uint32_t (&at)[kChainVec])
{
    StackTile<T, OP, BATCH>(d, src, ops, off, at, [&](uint32_t h, const auto &x) {
        constexpr uint32_t U = sizeof(x) / sizeof(V4);
        uint32_t where[U];
#pragma unroll
        for (uint32_t u = 0; u < U; u++) {
            where[u] = h == 0 ? pos[u] : pos[kChainVec - U + u];
        }
        StoreByFlags(d, dst, off, nbytes, where, x);
    });
}

template <typename T, int OP>
__device__ __forceinline__ void StackRest(const FusedDesc &d, bool ends, const void *const *__restrict__ src, const uint32_t *__restrict__ ops,
    void *const *__restrict__ dst)
{
    if (!ends) {
        const uint32_t n = RestBytes(d);
        if (n == 0) {
            return;
        }
        uint32_t pos[kChainVec], at[kChainVec];
        TilePositions(pos);
        ReadPositions(pos, n, at);
        StackStore<T, OP, kStackPlainBatch>(d, src, ops, dst, RestOffset(d), n, pos, at);
    } else {
        const uint32_t i = threadIdx.x * uint32_t(sizeof(T));
        if (i < EndBytes(d)) {
            const uint64_t off = EndOffset(d, i);
            const uint32_t at[1] = {0};
            T x[1];
            StackValue<ElemLane<T, OP>, T, OP, 1, true, 8>(d, src, ops, off, at, x);
            for (uint32_t k = 0; k < d.ndst; k++) {
                StoreElem<T>(dst[k], off, x[0]);
            }
        }
    }
}

template <typename T, int OP>
__global__ void __launch_bounds__(kBlockThreads) StackKernel(const FusedDesc *__restrict__ items, uint32_t nitems, uint32_t nall, uint32_t nwhole,
    uint32_t ntiles, const void *const *__restrict__ srcPool, void *const *__restrict__ dstPool, uint32_t tilesPerItem)
{
    const uint32_t *opPool = reinterpret_cast<const uint32_t *>(items + nall);
    uint32_t pos[kChainVec];
    TilePositions(pos);
    WalkTiles(items, nitems, nall, nwhole, ntiles, tilesPerItem, [](const FusedDesc &) { return 0; },
        [&](const FusedDesc &d, int, uint64_t off) {
            StackStore<T, OP, kStackPlainBatch>(d, srcPool + d.srcBase, opPool + d.srcBase, dstPool + d.dstBase, off, kTileBytes, pos, pos);
        },
        [&](const FusedDesc &d, bool ends) { StackRest<T, OP>(d, ends, srcPool + d.srcBase, opPool + d.srcBase, dstPool + d.dstBase); });
}

}  // namespace hcclamd

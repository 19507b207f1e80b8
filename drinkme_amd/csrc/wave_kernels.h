// The wave kernels: decode + GEMV (k_gemv_wave) and decode alone
// (k_decode_wave) for 1024-weight blocks of the three profiles, any column
// count, any activation type. They serve gulp at M <= 4 and what the sip and
// gulp kernels do not take: columns that are not whole blocks, the balanced
// profile, and fp32 activations. Included by kernels.hip, inside its namespace.
//
// Work split. A workgroup of W waves owns T rows (T even) of one tensor. A
// unit is one column block of two neighbouring rows; the units, column by
// column, are dealt to the waves in contiguous runs. So a wave stays on one
// column block for a run of rows and keeps that block's activations in
// registers, 16 columns a lane: they are read once per column block (from
// L2), not once per weight block, and cost no LDS traffic at any M. Each
// weight block's M sums are reduced over the lanes (both rows of the unit
// at once) into LDS, and a row's column blocks are added in order at the
// end. Every sum is a function of the row and the activation alone: the
// same for any M, T and W.
//
// What bounds it: for launches of a few units a wave, the 6 us before and
// after them (the directory's round trip, the first payload, the tables);
// for longer ones the decode: the VALU is busy 65% of the time (gulp, M = 1,
// 2 x 12288 x 4096; 70% at M = 4), 105 instructions a block (143) beside 60
// scalar and 18 LDS ones, and of a wave's life 37% issues (36%), 35% waits on a
// dependency (32%) and 28% for an issue slot (32%). (fp32 products are 16 M +
// 16 instructions a block more.) Measured, one launch, against k_gemv_generic, which scans over
// a workgroup with two barriers a tier: sip 2 x 9472 x 3584 (ragged) 21.2 us
// for 284, sip 3584 x 9472 14.3 for 149; gulp fp32 M = 2 q/k/v of 10240 x
// 5120 23.8 for 326; balanced q/k/v of 6144 x 4096 12.8 for 145. Against
// k_gemv_gulp: wave_first (kernels.hip). More waves measured slower at M = 1:
// 10-wave workgroups at five a SIMD 113 -> 139 us on the gulp MLP of 25600 x
// 5120, 12-wave ones at six (80 registers, spilled) 171.
//
// The decode works on bytes. A table entry holds the exponent bytes of the
// weights that resolved in this tier and a v_perm selector over (four
// consecutive bytes of the next tier's exponents, the entry's own four): byte
// k is 4 + the weight's rank among the group's e escapes, or e + its rank
// among the others (whose exponents lie at those bytes of the entry). One
// v_perm so completes a group, and with the own bytes placed so the bits set
// in the selector are 4 + e for every pattern: one popcount, unmasked, counts
// the escapes, and its 4 a group goes into the windows' immediate offsets.
//   tier 0   lane l owns weights 16l .. 16l + 15, four table lookups;
//   tier 1   (balanced, gulp) lane l resolves the block's tier-0 escapes
//            8l .. 8l + 7 from the tail words, which a wave keeps in LDS,
//            and writes their exponent bytes, in order, to LDS;
//   tier 2   (gulp) lane l resolves the tier-1 escapes 2l, 2l + 1 so;
//   terminal raw exponent bytes, read in place from the tail words.
// Each level reads the four bytes at its first escape's rank from the level
// below (two LDS words and a funnel shift). The ranks come from one DPP scan
// a level for both rows of a unit (counts of at most 1024, 16 bits each).
// The two rows' decodes run side by side with no branch between them, so one
// row's LDS round trips cover the other's (decoded one after the other, the
// waves waited 44% of their time). A block outside the limits (more than 512
// tier-0 or 128 tier-1 escapes, a tail of more than 64 words, streams cut
// short) takes wave_wide, which reads its streams from memory.

// Exponent bytes are kept rotated right by one: a byte's low seven bits are
// the bf16 high byte's and its top bit the low byte's, so merging them with
// the literals (sign and mantissa) takes one v_bfi a half.
__device__ __forceinline__ uint32_t rotate_bytes(uint32_t v) {
    return ((v >> 1) & 0x7F7F7F7Fu) | ((v << 7) & 0x80808080u);
}

// Two words of LDS from byte address `at` + `past` (a multiple of 4) on, `at`
// rounded down to a word, and the four bytes from `at` in them. (One unaligned ds_read_b32 instead
// stalls the LDS for about 60 cycles a wave: the 9472 x 3584 gate/up launch
// took 45.6 us with it, 28.8 us without.)
typedef const __attribute__((address_space(3))) uint32_t* lds_words;
__device__ __forceinline__ uint32_t lds_address(const void* p) { return (uint32_t)(uintptr_t)(lds_ptr)p; }
__device__ __forceinline__ uint2 lds_window(uint32_t at, uint32_t past = 0) {
    const lds_words p = (lds_words)(uintptr_t)(at & ~3u);
    return make_uint2(p[past / 4], p[past / 4 + 1]);
}
__device__ __forceinline__ uint32_t window_bytes(uint2 w, uint32_t at) { return __builtin_amdgcn_alignbyte(w.y, w.x, at); }

// Entry of N codes c[k] < 2^w (two: the selector's upper bytes are 0),
// exponents from the run `pal` of the padded tables.
template <uint32_t w, uint32_t N>
__device__ __forceinline__ uint2 wave_entry(uint32_t i, const uint32_t (&pal)[4]) {
    uint32_t e = 0, sel = 0, r = 4, own = 0;
#pragma unroll
    for (uint32_t k = 0; k < N; ++k) own += ((i >> (w * k)) & ((1u << w) - 1u)) == (1u << w) - 1u;
#pragma unroll
    for (uint32_t k = 0; k < N; ++k) {
        const uint32_t c = (i >> (w * k)) & ((1u << w) - 1u);
        uint32_t b = __builtin_amdgcn_perm(pal[1], pal[0], c & 7u);
        if (w == 4) b = c & 8u ? __builtin_amdgcn_perm(pal[3], pal[2], c & 7u) : b;
        const bool esc = c == (1u << w) - 1u;
        e |= esc ? 0u : (b & 0xFFu) << (8 * own);  // (rotated bytes, as pal's are)
        sel |= (esc ? r : own) << (8 * k);
        r += esc;
        own += !esc;
    }
    return make_uint2(e, sel);
}

// The 4096 entries of four 3-bit codes (palette words p0, p1): entries 8h ..
// 8h + 7 share the upper three codes, so but for c0 = 7 (an escape) their
// selector and the byte, `at`, of c0's exponent.
__device__ __forceinline__ void wave_table3(uint2* tab, uint32_t p0, uint32_t p1, uint32_t threads) {
    const uint32_t pal[4] = {p0, p1, 0, 0};
    for (uint32_t h = threadIdx.x; h < 512; h += threads) {
        const uint2 e = wave_entry<3, 4>(8 * h, pal), esc = wave_entry<3, 4>(8 * h + 7, pal);
        const uint32_t at = 8 * (e.y & 3u), up = e.x & ~(0xFFu << at);
#pragma unroll
        for (uint32_t c = 0; c < 8; c += 2) {
            const uint32_t two = c < 4 ? p0 >> (8 * c) : p1 >> (8 * (c - 4));
            const uint2 odd = c == 6 ? esc : make_uint2(up | ((two >> 8) & 0xFFu) << at, e.y);
            *reinterpret_cast<uint4*>(tab + 8 * h + c) = make_uint4(up | (two & 0xFFu) << at, e.y, odd.x, odd.y);
        }
    }
}

// Builds the tables of profile P (all of the workgroup's threads).
template <int P>
__device__ __forceinline__ void wave_tables(uint2* tab, const uint32_t* palette, uint32_t threads) {
    const const_u32_ptr pw = (const_u32_ptr)palette;
    auto p = [&](int i) { return rotate_bytes(pw[i]); };
    if constexpr (P == kWaveSip) {
        wave_table3(tab, p(0), p(1), threads);
    } else if constexpr (P == kWaveBalanced) {
        const uint32_t pal0[4] = {p(0), 0, 0, 0};
        for (uint32_t i = threadIdx.x; i < 256; i += threads) tab[i] = wave_entry<2, 4>(i, pal0);
        wave_table3(tab + 256, p(1), p(2), threads);
    } else if constexpr (P == kWaveGulp) {
        const uint32_t pal0[4] = {p(0), 0, 0, 0}, pal1[4] = {p(1), 0, 0, 0}, pal2[4] = {p(2), p(3), p(4), p(5)};
        for (uint32_t i = threadIdx.x; i < 768; i += threads)
            tab[i] = i < 256 ? wave_entry<2, 4>(i, pal0) : i < 512 ? wave_entry<2, 4>(i - 256, pal1)
                                                                  : wave_entry<4, 2>(i - 512, pal2);
    }
}

// A block's loads: the lane's 16 literal bytes, its tier-0 codes and its
// tail word (the streams after tier 0).
struct WaveStage {
    u32x4 lit;
    u32x2 t0;
    uint32_t tail;
};

// A block's size: n weights, lit words of literals, fixed words with tier 0.
struct BlockSize {
    uint32_t n, lit, fixed;
};
__device__ __forceinline__ BlockSize block_size(int P, uint32_t n) {
    return {n, words_for(n, 8), words_for(n, 8) + words_for(n, wave_width(P, 0))};
}

// Loads the block of len words at `start`, non-temporal, through a buffer
// resource that ends four words past the block (or its fixed streams, where
// the block is cut shorter than those): no wide load of a lane straddles the
// end, and those words are the next block's or the pad's. The tail's lanes
// past the block take an offset past the resource: they read 0 and fetch
// nothing. live = false: nothing is fetched. The loads are unconditional, so
// the compiler's waits for one stage leave the next one's loads in flight.
template <int P>
__device__ __forceinline__ WaveStage wave_load(const uint32_t* data, uint32_t start, int32_t len, const BlockSize& z,
                                               bool live, uint32_t lane) {
    const uint32_t reach = 4u * ((uint32_t)max(len, (int32_t)z.fixed) + 4u);
    const auto r = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>(data + start), 0, live ? reach : 0u, 0x00020000);
    constexpr int nt = 2;
    WaveStage s;
    s.lit = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, 16 * lane, 0, nt));
    if constexpr (P == kWaveSip) {
        s.t0 = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(r, 4 * (z.lit + ((3 * lane) >> 1)), 0, nt));
    } else {
        s.t0.x = __builtin_amdgcn_raw_buffer_load_b32(r, 4 * (z.lit + lane), 0, nt);
        s.t0.y = 0;
    }
    s.tail = __builtin_amdgcn_raw_buffer_load_b32(
        r, (int32_t)lane < len - (int32_t)z.fixed ? 4 * (z.fixed + lane) : 0x80000000u, 0, nt);
    return s;
}

// The first `bits` (clamped to 0 .. most < 32) bits of codes: those past the
// stream's end read as 0, which no tier takes for an escape.
__device__ __forceinline__ uint32_t keep_bits(uint32_t codes, int32_t bits, int32_t most) {
    return __builtin_amdgcn_ubfe(codes, 0, (uint32_t)min(max(bits, 0), most));
}

// Escapes of an entry of four codes, and 4 (of two codes, and 1), added to n.
__device__ __forceinline__ uint32_t add_escapes(uint2 e, uint32_t n) { return (uint32_t)__builtin_popcount(e.y) + n; }

// Completes an entry from the next tier's four exponent bytes.
__device__ __forceinline__ uint32_t complete(uint2 e, uint32_t next) { return __builtin_amdgcn_perm(next, e.x, e.y); }

// The farthest word past a block's start that any of its streams reaches.
constexpr uint32_t wave_bound(int P) {
    uint32_t b = 2 * 256;  // literals, terminal
    for (uint32_t j = 0; j < wave_tiers(P); ++j) b += 32 * wave_width(P, j);
    return b;
}

// The lane's 16 exponent bytes (rotated) of a block outside the limits, with
// the meaning of decode_block: any escape counts, streams of any length, read
// from memory. Lane l owns codes 16l .. 16l + 15 of every tier, two words of
// them at most, so a tier costs one round trip to memory (tier 0 and tier 1
// together: their places are known), its lookups and one scan; each level's
// bytes go down through the exchange, whose first 258 words serve the levels
// in turn, and the terminal's are read in place. Such blocks are ordinary
// where one palette serves rows of different scale: of 12288 x 4096 N(0, 0.02)
// gulp weights with rows scaled by a lognormal of sigma 0.3, 0.5, 1.0, M = 1,
// the launch takes 22, 27, 43 us (unscaled 18); reading one field at a time,
// both rows of a unit together, took 78, 142, 226. The loads go through a
// buffer resource that ends one word past the streams' bound, which the pad
// covers: the bound counts from the block's first word.
template <int P>
__device__ __forceinline__ void wave_wide(const uint2* tab, uint32_t* ex, const uint32_t* data, uint32_t start,
                                          uint32_t end, const BlockSize& z, uint32_t lane, uint32_t (&E)[4]) {
    const auto r = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>(data + start), 0, 4 * (wave_bound(P) + 1),
                                                     0x00020000);
    const uint32_t len = end - start;
    uint32_t pos = z.fixed;
    asm volatile("" : "+v"(lane));  // (else its multiples are kept in registers over the unit loop)
    auto words = [&](uint32_t byte) {  // two words of the block, from the byte on (a multiple of 4)
        return __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(r, byte, 0, 0));
    };
    auto load = [&](uint32_t at, uint32_t n, uint32_t w, uint32_t (&t)[2]) {  // 16 w-bit codes of n at word `at`
        const uint32_t bit = 16 * w * lane;
        const u32x2 v = words(16 * lane < n ? 4 * (at + (bit >> 5)) : 0x80000000u);
        const uint64_t all = ((uint64_t)v.y << 32 | v.x) >> (bit & 31u);
        t[0] = (uint32_t)all;
        t[1] = (uint32_t)(all >> 32);
    };
    auto keep = [&](uint32_t n, uint32_t w, uint32_t (&t)[2]) {
        const int32_t bits = ((int32_t)n - 16 * (int32_t)lane) * (int32_t)w;
        t[0] = bits >= 32 ? t[0] : keep_bits(t[0], bits, 31);
        t[1] = bits >= 64 ? t[1] : keep_bits(t[1], bits - 32, 31);
    };
    auto group = [&](const uint2* t, uint32_t w, const uint32_t (&c)[2], int g) {  // four codes' entry
        const uint64_t v = (uint64_t)c[1] << 32 | c[0];
        return t[(uint32_t)(v >> (4 * w * g)) & ((1u << (4 * w)) - 1u)];
    };
    // the rank of the lane's first escape among a tier's (four groups of codes
    // c), and how many there are
    auto scan = [&](uint32_t cnt, uint32_t& first, uint32_t& total) {
        const uint32_t inc = wave_scan_incl_dpp(cnt);
        first = inc - cnt;
        total = __builtin_amdgcn_readlane(inc, 63);
    };
    auto escapes = [&](const uint2* t, uint32_t w, const uint32_t (&c)[2]) {
        uint32_t n = 0;
#pragma unroll
        for (int g = 0; g < 4; ++g) n += add_escapes(group(t, w, c, g), ~3u);
        return n;
    };
    // the four groups' bytes, completed by those `next` gives from a rank on
    // (the entries looked up again: kept over the tiers below, they spill)
    auto resolve = [&](const uint2* t, uint32_t w, const uint32_t (&c)[2], uint32_t q, auto next, uint32_t (&v)[4]) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const uint2 en = group(t, w, c, g);
            v[g] = complete(en, next(q));
            q += add_escapes(en, ~3u);
        }
    };
    const uint32_t ex_at = lds_address(ex);
    auto terminal = [&](uint32_t q) {  // (read only where the directory gives the block words for it)
        if (len <= pos) return 0u;
        const u32x2 v = words(4 * pos + (q & ~3u));
        return rotate_bytes(window_bytes(make_uint2(v.x, v.y), q));
    };
    auto below = [&](uint32_t q) { return window_bytes(lds_window(ex_at + q), q); };  // (ex_at is a whole word's)
    auto put = [&](const uint32_t (&v)[4]) {
#pragma unroll
        for (int g = 0; g < 4; ++g) ex[4 * lane + g] = v[g];
        wave_lds_sync();
    };
    constexpr uint32_t w0 = wave_width(P, 0), w1 = wave_width(P, 1);
    uint32_t t0[2], q0, n1;
    load(z.lit, z.n, w0, t0);
    if constexpr (P == kWaveSip) {
        keep(z.n, w0, t0);
        scan(escapes(tab, w0, t0), q0, n1);
        resolve(tab, w0, t0, q0, terminal, E);
    } else {
        uint32_t t1[2], q1, n2, v[4];
        load(pos, 1024, w1, t1);
        keep(z.n, w0, t0);
        scan(escapes(tab, w0, t0), q0, n1);
        pos += words_for(n1, w1);
        keep(n1, w1, t1);
        scan(escapes(tab + 256, w1, t1), q1, n2);
        if constexpr (P == kWaveBalanced) {
            resolve(tab + 256, w1, t1, q1, terminal, v);
        } else {
            uint32_t t2[2], q2, n3, cnt = 0;
            load(pos, n2, 4, t2);
            keep(n2, 4, t2);
            auto pair = [&](int i) { return tab[512 + ((t2[i / 4] >> (8 * (i & 3))) & 0xFFu)]; };
#pragma unroll
            for (int i = 0; i < 8; ++i) cnt += add_escapes(pair(i), ~0u);
            scan(cnt, q2, n3);
            pos += words_for(n2, 4);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const uint2 en = pair(i);
                const uint32_t two = (n3 ? complete(en, terminal(q2)) : en.x) & 0xFFFFu;
                q2 += add_escapes(en, ~0u);
                v[i / 2] = i & 1 ? v[i / 2] | two << 16 : two;
            }
            put(v);
            resolve(tab + 256, w1, t1, q1, below, v);
            wave_lds_sync();
        }
        put(v);
        resolve(tab, w0, t0, q0, below, E);
        wave_lds_sync();
    }
}

// Decodes R blocks of size z (R = 2: a unit's rows; 1) from their loaded
// stages: hi[j][g], lo[j][g] = the high and low bytes of the bf16 bits of the
// lane's weights 4g .. 4g + 3 of block j (weight k in byte k). Weights past
// the block get exponent 0 (a zero or denormal, finite: their activations
// are 0). ex: the wave's exchange, R x wave_exchange(P) words, in front of
// the tables, so that a block outside the limits, whose window addresses
// reach at most 1 KB too far, still reads inside the LDS array. The
// sched_barriers keep a level's LDS reads together: left to itself the
// compiler waits for each before it issues the next.
template <int P, int R>
__device__ __forceinline__ void wave_decode(const uint2* tab, uint32_t* ex, const WaveStage (&s)[R], const uint32_t* data,
                                            const uint32_t (&start)[R], const int32_t (&len)[R], const BlockSize& z,
                                            uint32_t lane, uint32_t (&hi)[R][4], uint32_t (&lo)[R][4]) {
    constexpr uint32_t stride = wave_exchange(P);
    const uint32_t ex_at = lds_address(ex);
    uint2 e[R][4];
    uint32_t c[R][4];  // escapes of groups 0 .. g, less 4 (3 - g)
    int32_t tail[R], bad[R];  // (bad: negative once a limit is passed; every quantity is far below 2^31)
    uint32_t T[R][2];
#pragma unroll
    for (int j = 0; j < R; ++j) {
        tail[j] = len[j] - (int32_t)z.fixed;
        bad[j] = 64 - tail[j];
        ex[j * stride + kExTerm + lane] = rotate_bytes(s[j].tail);
        if constexpr (P != kWaveSip) ex[j * stride + kExTail + lane] = s[j].tail;
        if constexpr (P == kWaveSip) {
            const uint64_t v = ((uint64_t)s[j].t0.y << 32 | s[j].t0.x) >> ((lane & 1) * 16);
            T[j][0] = (uint32_t)v;
            T[j][1] = (uint32_t)(v >> 32);
        } else {
            T[j][0] = s[j].t0.x;
        }
    }
    wave_lds_sync();
    if (z.n < 1024) {
        const int32_t bits = ((int32_t)z.n - 16 * (int32_t)lane) * (int32_t)wave_width(P, 0);
#pragma unroll
        for (int j = 0; j < R; ++j) {
            T[j][0] = bits >= 32 ? T[j][0] : keep_bits(T[j][0], bits, 31);
            if constexpr (P == kWaveSip) T[j][1] = keep_bits(T[j][1], bits - 32, 16);
        }
    }
#pragma unroll
    for (int j = 0; j < R; ++j) {
        if constexpr (P == kWaveSip) {
            e[j][0] = tab[T[j][0] & 0xFFFu];
            e[j][1] = tab[(T[j][0] >> 12) & 0xFFFu];
            e[j][2] = tab[__builtin_amdgcn_alignbit(T[j][1], T[j][0], 24) & 0xFFFu];
            e[j][3] = tab[(T[j][1] >> 4) & 0xFFFu];
        } else {
#pragma unroll
            for (int g = 0; g < 4; ++g) e[j][g] = tab[(T[j][0] >> (8 * g)) & 0xFFu];
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    // counts of both rows through one scan, row j in bits 16j .. 16j + 15
    uint32_t q[R], n1[R];
    auto scan = [&](const uint32_t (&cnt)[R], uint32_t (&first)[R], uint32_t (&total)[R]) {
        const uint32_t v = R == 2 ? cnt[0] | cnt[R - 1] << 16 : cnt[0];
        const uint32_t inc = wave_scan_incl_dpp(v), x = inc - v, t = __builtin_amdgcn_readlane(inc, 63);
        first[0] = R == 2 ? x & 0xFFFFu : x;
        total[0] = R == 2 ? t & 0xFFFFu : t;
        if (R == 2) {
            first[R - 1] = x >> 16;
            total[R - 1] = t >> 16;
        }
    };
    uint32_t cnt[R];
#pragma unroll
    for (int j = 0; j < R; ++j) {
        c[j][0] = add_escapes(e[j][0], ~15u);
#pragma unroll
        for (int g = 1; g < 4; ++g) c[j][g] = add_escapes(e[j][g], c[j][g - 1]);
        cnt[j] = c[j][3];
    }
    scan(cnt, q, n1);
    uint32_t below = kExTerm;  // where tier 0's escapes lie, in words of the exchange
    if constexpr (P == kWaveSip) {
#pragma unroll
        for (int j = 0; j < R; ++j) bad[j] |= 4 * tail[j] - (int32_t)n1[j];
    } else {
        // lane l: the block's tier-1 codes 8l .. 8l + 7
        constexpr uint32_t w = wave_width(P, 1);
        uint32_t w1[R], g0[R], q1[R], n2[R];  // (g0: escapes of the first group, less 4)
        uint2 a[R][2];
        uint2 win[R][2];
        // the two groups' windows in the exponent bytes at byte `at` of the
        // exchange, and the groups completed from them
        uint32_t p1[R];
        auto windows = [&](int j, uint32_t at) {
            p1[j] = q1[j] + at;
            win[j][0] = lds_window(p1[j]);
            win[j][1] = lds_window(p1[j] + g0[j], 4);
        };
        auto finish = [&]() {
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < R; ++j) {
                a[j][0].x = complete(a[j][0], window_bytes(win[j][0], p1[j]));
                a[j][1].x = complete(a[j][1], window_bytes(win[j][1], p1[j] + g0[j]));
            }
        };
#pragma unroll
        for (int j = 0; j < R; ++j) {
            const uint32_t t = ex_at + 4 * (j * stride + kExTail);
            w1[j] = words_for(n1[j], w);
            const int32_t bits = (int32_t)(w * n1[j]) - (int32_t)(8 * w * lane);
            if constexpr (P == kWaveBalanced) {
                const uint32_t code = keep_bits(window_bytes(lds_window(t + 3 * lane), 3 * lane), bits, 24);
                a[j][0] = tab[256 + (code & 0xFFFu)];
                a[j][1] = tab[256 + (code >> 12)];
            } else {
                const uint32_t code =
                    keep_bits(reinterpret_cast<const uint16_t*>(ex + j * stride + kExTail)[lane], bits, 16);
                a[j][0] = tab[256 + (code & 0xFFu)];
                a[j][1] = tab[256 + (code >> 8)];
            }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < R; ++j) {
            g0[j] = add_escapes(a[j][0], ~7u);
            cnt[j] = add_escapes(a[j][1], g0[j]);
        }
        scan(cnt, q1, n2);
        if constexpr (P == kWaveBalanced) {
#pragma unroll
            for (int j = 0; j < R; ++j) {
                const int32_t left = tail[j] - (int32_t)w1[j];  // terminal words
                bad[j] |= (512 - (int32_t)n1[j]) | left | (4 * left - (int32_t)n2[j]);
                windows(j, ex_at + 4 * (j * stride + kExTerm + (w1[j] & 63u)));
            }
        } else {
            // lane l: the block's tier-2 codes 2l, 2l + 1
            uint2 b[R];
            uint32_t w2[R];
#pragma unroll
            for (int j = 0; j < R; ++j) {
                w2[j] = words_for(n2[j], 4);
                const uint32_t code = reinterpret_cast<const uint8_t*>(ex + j * stride + kExTail + (w1[j] & 63u))[lane];
                b[j] = tab[512 + keep_bits(code, (int32_t)(4 * n2[j]) - (int32_t)(8 * lane), 8)];
                bad[j] |= (512 - (int32_t)n1[j]) | (128 - (int32_t)n2[j]) | (tail[j] - (int32_t)(w1[j] + w2[j]));
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < R; ++j) cnt[j] = add_escapes(b[j], ~0u);
            if (__builtin_amdgcn_ballot_w64((cnt[0] | cnt[R - 1]) != 0) != 0) {
                uint32_t q2[R], n3[R];
                scan(cnt, q2, n3);
#pragma unroll
                for (int j = 0; j < R; ++j) {
                    bad[j] |= 4 * (tail[j] - (int32_t)(w1[j] + w2[j])) - (int32_t)n3[j];
                    const uint32_t at = ex_at + 4 * (j * stride + kExTerm + ((w1[j] + w2[j]) & 63u)) + q2[j];
                    b[j].x = complete(b[j], window_bytes(lds_window(at), at));
                }
            }
#pragma unroll
            for (int j = 0; j < R; ++j) reinterpret_cast<uint16_t*>(ex + j * stride + kExT2)[lane] = (uint16_t)b[j].x;
            wave_lds_sync();
#pragma unroll
            for (int j = 0; j < R; ++j) windows(j, ex_at + 4 * (j * stride + kExT2));
        }
        finish();
#pragma unroll
        for (int j = 0; j < R; ++j)
            *reinterpret_cast<uint2*>(ex + j * stride + kExT1 + 2 * lane) = make_uint2(a[j][0].x, a[j][1].x);
        wave_lds_sync();
        below = kExT1;
    }
    uint2 win[R][4];
#pragma unroll
    for (int j = 0; j < R; ++j) {
        q[j] += ex_at + 4 * (j * stride + below);
        win[j][0] = lds_window(q[j]);
#pragma unroll
        for (int g = 1; g < 4; ++g) win[j][g] = lds_window(c[j][g - 1] += q[j], 16 - 4 * g);
    }
    __builtin_amdgcn_sched_barrier(0);
    uint32_t E[R][4];
#pragma unroll
    for (int j = 0; j < R; ++j) {
        E[j][0] = complete(e[j][0], window_bytes(win[j][0], q[j]));
#pragma unroll
        for (int g = 1; g < 4; ++g) E[j][g] = complete(e[j][g], window_bytes(win[j][g], c[j][g - 1]));
    }
    wave_lds_sync();
    if (__builtin_expect((bad[0] | bad[R - 1]) < 0, 0)) {
#pragma unroll 1
        for (int j = 0; j < R; ++j) {
            if ((j ? bad[R - 1] : bad[0]) >= 0) continue;
            uint32_t x[4];
            const uint32_t at = j ? start[R - 1] : start[0];
            wave_wide<P>(tab, ex, data, at, at + (uint32_t)(j ? len[R - 1] : len[0]), z, lane, x);
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                E[0][g] = j == 0 ? x[g] : E[0][g];
                E[R - 1][g] = j == R - 1 ? x[g] : E[R - 1][g];
            }
        }
    }
    if (z.n < 1024) {
        const int32_t valid = (int32_t)z.n - 16 * (int32_t)lane;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const uint32_t keep = valid >= 4 * g + 4 ? ~0u : keep_bits(~0u, 8 * (valid - 4 * g), 24);
#pragma unroll
            for (int j = 0; j < R; ++j) E[j][g] &= keep;
        }
    }
#pragma unroll
    for (int j = 0; j < R; ++j)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const uint32_t L = s[j].lit[g];
            hi[j][g] = (L & 0x80808080u) | (E[j][g] & 0x7F7F7F7Fu);
            lo[j][g] = (L & 0x7F7F7F7Fu) | (E[j][g] & 0x80808080u);
        }
}

// The lane's pair words (weights 16l + 2i, + 1) of a decoded block.
__device__ __forceinline__ void wave_pairs(const uint32_t (&hi)[4], const uint32_t (&lo)[4], uint32_t (&wp)[8]) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        wp[2 * g] = __builtin_amdgcn_perm(hi[g], lo[g], 0x05010400u);
        wp[2 * g + 1] = __builtin_amdgcn_perm(hi[g], lo[g], 0x07030602u);
    }
}

// ---- sums over the lanes

template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}
// Lanes 0..31: a summed over lanes l, l + 32; lanes 32..63: b so.
__device__ __forceinline__ float fold32(float a, float b) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// The same over rows of 16 lanes: even rows a (l, l + 16), odd rows b.
__device__ __forceinline__ float fold16(float a, float b) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// Lanes with `bit` clear: a plus its partner's a; with it set: b so.
template <int CTRL>
__device__ __forceinline__ float fold_dpp(float a, float b, bool bit) {
    const float keep = bit ? b : a, give = bit ? a : b;
    return keep + dpp_move<CTRL>(give);
}

// V values (2..16) summed over the 64 lanes: value i in the lanes with
// lane / (64 / V) == i. The tree is the same for every V: partners at lane
// distance 32, 16 and 8, the mirror within 8, then 2 and 1.
template <int V>
__device__ __forceinline__ float wave_fold(float (&v)[V], uint32_t lane) {
    constexpr int V1 = V / 2, V2 = V1 > 1 ? V1 / 2 : 1, V3 = V2 > 1 ? V2 / 2 : 1;
#pragma unroll
    for (int i = 0; i < V1; ++i) v[i] = fold32(v[i], v[i + V1]);
#pragma unroll
    for (int i = 0; i < V2; ++i) v[i] = fold16(v[i], v[V1 > 1 ? i + V2 : i]);
#pragma unroll
    for (int i = 0; i < V3; ++i) v[i] = V2 > 1 ? fold_dpp<0x128>(v[i], v[i + V3], lane & 8u) : v[i] + dpp_move<0x128>(v[i]);
    float s = V3 > 1 ? fold_dpp<0x141>(v[0], v[V3 > 1 ? 1 : 0], lane & 4u) : v[0] + dpp_move<0x141>(v[0]);
    s += dpp_move<0x4E>(s);
    return s + dpp_move<0xB1>(s);
}

// ---- decode + GEMV

struct WaveGroup {
    const uint32_t* data[kGroupMax];  // the raw weight in kWaveRaw
    const uint32_t* offsets[kGroupMax];
    const uint32_t* palette[kGroupMax];
    const void* bias[kGroupMax];
    void* out[kGroupMax];
    uint32_t rows[kGroupMax];
    uint32_t wg0[kGroupMax + 1];  // tensor i's workgroups: wg0[i] .. wg0[i + 1] - 1
};

struct WaveShape {
    uint32_t cols, nb;
    uint32_t tile;  // T: rows per workgroup, even
    uint32_t m;     // activation rows (<= the kernel's M; the rest repeat the last one)
    uint32_t wide;  // 1: x's rows (raw: the weight's too) may be read four bytes at a time
    int bias_dtype, out_dtype;
};

struct __attribute__((packed, aligned(4))) Quad4 {
    uint32_t v[4];
};

constexpr uint32_t kDecodeWaves = 8;
template <int P, int M, int XT>
__global__ __launch_bounds__(wave_waves(P, M, XT) * 64, wave_occ(P, M, XT))
void k_gemv_wave(const WaveGroup g, const void* __restrict__ x, const WaveShape sh) {
    constexpr uint32_t W = wave_waves(P, M, XT);
    constexpr int XR = XT == kWaveX32 ? 16 : 8;  // activation registers per row
    __shared__ __align__(16) uint2 lds[kExHead + W * wave_exchange(P) + wave_entries(P)];
    uint2* tab = lds + kExHead + W * wave_exchange(P);
    extern __shared__ __align__(16) uint8_t lds_dyn[];
    float* red = reinterpret_cast<float*>(lds_dyn);

    const uint32_t wv = wave_id(), lane = lane_id();
    uint32_t it = 0;
#pragma unroll
    for (int i = 1; i < kGroupMax; ++i) it += blockIdx.x >= g.wg0[i];
    const uint32_t* data = pick(g.data, it);
    const uint32_t* offsets = pick(g.offsets, it);
    const uint32_t* palette = pick(g.palette, it);
    const uint32_t rows = pick(g.rows, it);
    uint32_t wg0 = g.wg0[0];
#pragma unroll
    for (int i = 1; i < kGroupMax; ++i) wg0 = it == (uint32_t)i ? g.wg0[i] : wg0;
    const uint32_t r0 = (blockIdx.x - wg0) * sh.tile, nrows = min(sh.tile, rows - r0);
    const uint32_t pairs = (nrows + 1) / 2, units = pairs * sh.nb;
    const uint32_t u0 = units * wv / W, u1 = units * (wv + 1) / W;
    const uint32_t first = r0 * sh.nb;  // the tile's first block
    uint32_t* ex0 = reinterpret_cast<uint32_t*>(lds + kExHead) + wv * 2 * wave_exchange(P);

    uint32_t xr[M][XR];
    // (through one buffer resource, a row's start the scalar offset: 128-bit
    // loads in a whole block; in the last, partial one a dword each, or an
    // element where the rows are not dword-aligned, and a lane past the row
    // takes an offset past the resource: it reads 0 and fetches nothing)
    const auto rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(x), 0, 0x7FFFFFFF, 0x00020000);
    auto load_x = [&](uint32_t cb) {
        const uint32_t c0 = cb * 1024 + 16 * lane;
        constexpr uint32_t size = XT == kWaveX32 ? 4 : 2, per = 4 / size;  // elements a register
        auto at = [&](uint32_t c) { return c < sh.cols ? c * size : 0x80000000u; };
        if (sh.wide && cb * 1024 + 1024 <= sh.cols) {
#pragma unroll
            for (int m = 0; m < M; ++m)
#pragma unroll
                for (int i = 0; i < XR / 4; ++i) {
                    const auto v = __builtin_amdgcn_raw_buffer_load_b128(
                        rx, c0 * size + 16 * i, min((uint32_t)m, sh.m - 1) * sh.cols * size, 0);
#pragma unroll
                    for (int k = 0; k < 4; ++k) xr[m][4 * i + k] = v[k];
                }
        } else if (XT == kWaveX32 || sh.wide) {
#pragma unroll
            for (uint32_t i = 0; i < XR; ++i) {
                const uint32_t o = at(c0 + per * i);
#pragma unroll
                for (int m = 0; m < M; ++m)
                    xr[m][i] = __builtin_amdgcn_raw_buffer_load_b32(rx, o, min((uint32_t)m, sh.m - 1) * sh.cols * size, 0);
            }
        } else {
#pragma unroll
            for (uint32_t i = 0; i < XR; ++i) {
                const uint32_t o = at(c0 + 2 * i), o1 = at(c0 + 2 * i + 1);
#pragma unroll
                for (int m = 0; m < M; ++m) {
                    const uint32_t row = min((uint32_t)m, sh.m - 1) * sh.cols * size;
                    xr[m][i] = (uint32_t)(uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rx, o, row, 0) |
                               (uint32_t)(uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rx, o1, row, 0) << 16;
                }
            }
        }
    };
    // the activations waited on here, so that no later use of them waits on
    // loads issued after
    auto pin_x = [&]() {
#pragma unroll
        for (int m = 0; m < M; ++m)
#pragma unroll
            for (int i = 0; i < XR; ++i) asm volatile("" : "+v"(xr[m][i]));
    };

    // the directory entries of the next 32 units, one block a lane
    uint32_t o_start = 0, o_end = 0;
    auto load_directory = [&](uint32_t u) {
        if constexpr (P != kWaveRaw) {
            const uint32_t uu = min(u + (lane >> 1), u1 - 1), cb = uu / pairs, pr = uu - cb * pairs;
            const uint32_t blk = first + min(2 * pr + (lane & 1u), nrows - 1) * sh.nb + cb;
            o_start = offsets[blk];
            o_end = offsets[blk + 1];
        }
    };
    constexpr int SP = P == kWaveRaw ? kWaveSip : P;  // (the raw weight has no streams: sizes unused)
    const BlockSize whole = block_size(SP, 1024), last = block_size(SP, sh.cols - (sh.nb - 1) * 1024);
    auto size_of = [&](uint32_t cb) {
        const bool l = cb + 1 == sh.nb;
        return BlockSize{l ? last.n : whole.n, l ? last.lit : whole.lit, l ? last.fixed : whole.fixed};
    };
    struct Unit {
        WaveStage s[2];
        uint32_t start[2];
        int32_t len[2];
    };
    auto load_unit = [&](Unit& t, uint32_t k, uint32_t cb, bool live) {
        if constexpr (P != kWaveRaw) {
            const BlockSize z = size_of(cb);
#pragma unroll
            for (uint32_t j = 0; j < 2; ++j) {
                t.start[j] = __builtin_amdgcn_readlane(o_start, 2 * k + j);
                t.len[j] = (int32_t)(__builtin_amdgcn_readlane(o_end, 2 * k + j) - t.start[j]);
                t.s[j] = wave_load<P>(data, t.start[j], t.len[j], z, live, lane);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    // where the lane's folded sum goes: value i = lane / span is row i / M of
    // the unit, activation row i % M
    constexpr uint32_t span = 64 / (2 * M);
    float* const red_lane = red + (lane / span / M * sh.nb * M + lane / span % M);
    auto process = [&](const Unit& t, uint32_t cb, uint32_t pr) {
        float v[2 * M];
        uint32_t hi2[2][4], lo2[2][4];
        if constexpr (P != kWaveRaw)
            wave_decode<P, 2>(tab, ex0, t.s, data, t.start, t.len, size_of(cb), lane, hi2, lo2);
#pragma unroll
        for (uint32_t j = 0; j < 2; ++j) {
            uint32_t wp[8];
            const uint32_t(&hi)[4] = hi2[j], (&lo)[4] = lo2[j];
            if constexpr (P == kWaveRaw) {
                const uint32_t c0 = cb * 1024 + 16 * lane, n = sh.cols > c0 ? min(16u, sh.cols - c0) : 0u;
                const uint16_t* w = reinterpret_cast<const uint16_t*>(data) +
                                    (uint64_t)(r0 + min(2 * pr + j, nrows - 1)) * sh.cols + c0;
                if (cb * 1024 + 1024 <= sh.cols && (reinterpret_cast<uintptr_t>(data) & 15u) == 0 && sh.cols % 8 == 0) {
                    const u32x4 q0 = reinterpret_cast<const u32x4*>(w)[0], q1 = reinterpret_cast<const u32x4*>(w)[1];
#pragma unroll
                    for (uint32_t i = 0; i < 8; ++i) wp[i] = i < 4 ? q0[i & 3] : q1[i & 3];
                } else {
#pragma unroll
                    for (uint32_t i = 0; i < 8; ++i)
                        wp[i] = (2 * i < n ? (uint32_t)w[2 * i] : 0u) | (2 * i + 1 < n ? (uint32_t)w[2 * i + 1] << 16 : 0u);
                }
            }
            if constexpr (XT == kWaveX32) {
                float w[16];
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    if constexpr (P == kWaveRaw)
                        w[i] = __uint_as_float(i & 1 ? wp[i / 2] & 0xFFFF0000u : wp[i / 2] << 16);
                    else
                        w[i] = __uint_as_float(__builtin_amdgcn_perm(hi[i / 4], lo[i / 4], ((4u + i % 4) << 24) | ((i % 4) << 16) | 0x0C0Cu));
                }
#pragma unroll
                for (int m = 0; m < M; ++m) {
                    float a = w[0] * __uint_as_float(xr[m][0]), b = w[1] * __uint_as_float(xr[m][1]);
#pragma unroll
                    for (int i = 2; i < 16; i += 2) {
                        a = fmaf(w[i], __uint_as_float(xr[m][i]), a);
                        b = fmaf(w[i + 1], __uint_as_float(xr[m][i + 1]), b);
                    }
                    v[j * M + m] = a + b;
                }
            } else {
                if constexpr (P != kWaveRaw) wave_pairs(hi, lo, wp);
#pragma unroll
                for (int m = 0; m < M; ++m) {
                    float a = dot2(wp[0], xr[m][0], 0.0f), b = dot2(wp[1], xr[m][1], 0.0f);
#pragma unroll
                    for (int i = 2; i < 8; i += 2) {
                        a = dot2(wp[i], xr[m][i], a);
                        b = dot2(wp[i + 1], xr[m][i + 1], b);
                    }
                    v[j * M + m] = a + b;
                }
            }
        }
        const float s = wave_fold<2 * M>(v, lane);
        if (lane % span == 0) red_lane[(2 * pr * sh.nb + cb) * M] = s;
    };

    if (u0 < u1) load_directory(u0);
    uint32_t cb = u0 / pairs, pr = u0 - cb * pairs;
    Unit a, b;
    load_unit(a, 0, cb, u0 < u1);
    load_x(min(cb, sh.nb - 1));
    wave_tables<P>(tab, palette, W * 64);
    __syncthreads();
    pin_x();
    // unit k of the run is in flight (in a or b) when its turn comes; its
    // successor's loads are issued first
    for (uint32_t u = u0; u < u1;) {
        const uint32_t n = min(32u, u1 - u);
        for (uint32_t k = 0; k < n; k += 2) {
            uint32_t pr1 = pr + 1, cb1 = cb;
            if (pr1 == pairs) pr1 = 0, ++cb1;
            load_unit(b, (k + 1) & 31u, min(cb1, sh.nb - 1), k + 1 < n);
            process(a, cb, pr);
            if (k + 1 < n && cb1 != cb) {
                load_x(cb1);
                pin_x();
            }
            uint32_t pr2 = pr1 + 1, cb2 = cb1;
            if (pr2 == pairs) pr2 = 0, ++cb2;
            load_unit(a, (k + 2) & 31u, min(cb2, sh.nb - 1), k + 2 < n);
            if (k + 1 < n) process(b, cb1, pr1);
            cb = cb2, pr = pr2;
            if (k + 2 < n && cb2 != cb1) {
                load_x(cb2);
                pin_x();
            }
        }
        u += n;
        if (u < u1) {  // (n was 32: cb, pr are unit u's)
            load_directory(u);
            load_unit(a, 0, cb, true);
            load_x(cb);
            pin_x();
        }
    }
    __syncthreads();
    const void* bias = pick(g.bias, it);
    void* out = pick(g.out, it);
    for (uint32_t i = threadIdx.x; i < nrows * sh.m; i += W * 64) {
        const uint32_t m = i / nrows, t = i - m * nrows;
        float sum = 0.0f;
        for (uint32_t c = 0; c < sh.nb; ++c) sum += red[(t * sh.nb + c) * M + m];
        if (bias) sum += load_elem(bias, sh.bias_dtype, r0 + t);
        store_elem(out, sh.out_dtype, (uint64_t)m * rows + r0 + t, sum);
    }
}

// ---- decode

// Every block to its bf16 bits: a wave takes `run` consecutive blocks (at
// most 64, whose directory entries its lanes hold), the next one's loads in
// flight while it decodes and stores one. wide: the output's rows may be
// written four bytes at a time.
template <int P>
__global__ __launch_bounds__(kDecodeWaves * 64, 4) void k_decode_wave(Desc d, uint16_t* __restrict__ out, uint32_t run,
                                                                     uint32_t wide) {
    constexpr uint32_t W = kDecodeWaves;
    __shared__ __align__(16) uint2 lds[kExHead + W * wave_exchange(P) / 2 + wave_entries(P)];
    uint2* tab = lds + kExHead + W * wave_exchange(P) / 2;
    const uint32_t wv = wave_id(), lane = lane_id(), blocks = d.rows * d.nb;
    const uint32_t b0 = min(blocks, (blockIdx.x * W + wv) * run), n = min(run, blocks - b0);
    uint32_t* ex = reinterpret_cast<uint32_t*>(lds + kExHead) + wv * wave_exchange(P);
    uint32_t o_start = 0, o_end = 0;
    if (lane < n) {
        o_start = d.offsets[b0 + lane];
        o_end = d.offsets[b0 + lane + 1];
    }
    auto size_of = [&](uint32_t c) { return block_size(P, min(1024u, d.cols - c * 1024)); };
    auto load = [&](uint32_t k, uint32_t c, bool live) {
        const uint32_t start = __builtin_amdgcn_readlane(o_start, k & 63u);
        const WaveStage s = wave_load<P>(d.data, start, (int32_t)(__builtin_amdgcn_readlane(o_end, k & 63u) - start),
                                         size_of(c), live, lane);
        __builtin_amdgcn_sched_barrier(0);
        return s;
    };
    auto finish = [&](const WaveStage& s, uint32_t k, uint32_t row, uint32_t c) {
        uint32_t hi[1][4], lo[1][4], wp[8];
        const BlockSize z = size_of(c);
        const uint32_t w = z.n;
        const WaveStage st[1] = {s};
        const uint32_t start[1] = {(uint32_t)__builtin_amdgcn_readlane(o_start, k)};
        const int32_t len[1] = {(int32_t)(__builtin_amdgcn_readlane(o_end, k) - start[0])};
        wave_decode<P, 1>(tab, ex, st, d.data, start, len, z, lane, hi, lo);
        wave_pairs(hi[0], lo[0], wp);
        uint16_t* dst = out + (uint64_t)row * d.cols + c * 1024 + 16 * lane;
        if (wide && 16 * lane + 16 <= w) {
            reinterpret_cast<Quad4*>(dst)[0] = Quad4{{wp[0], wp[1], wp[2], wp[3]}};
            reinterpret_cast<Quad4*>(dst)[1] = Quad4{{wp[4], wp[5], wp[6], wp[7]}};
        } else {
#pragma unroll
            for (uint32_t i = 0; i < 16; ++i)
                if (16 * lane + i < w) dst[i] = (uint16_t)(wp[i / 2] >> (16 * (i & 1)));
        }
    };
    uint32_t row = b0 / d.nb, c = b0 - row * d.nb;
    WaveStage a = load(0, c, n != 0), b;
    wave_tables<P>(tab, reinterpret_cast<const uint32_t*>(d.table), W * 64);
    __syncthreads();
    for (uint32_t k = 0; k < n; k += 2) {
        uint32_t row1 = row, c1 = c + 1;
        if (c1 == d.nb) c1 = 0, ++row1;
        b = load(k + 1, c1, k + 1 < n);
        finish(a, k, row, c);
        row = row1, c = c1 + 1;
        if (c == d.nb) c = 0, ++row;
        a = load(k + 2, c, k + 2 < n);
        if (k + 1 < n) finish(b, k + 1, row1, c1);
    }
}

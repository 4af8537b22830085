// Tiling and factorisation heuristics for the gfx950 kernels.
// Plays the role of the reference's configure_small_batch_fft / configure_factor2_slm_fft
// (src/base/generator/small_batch_fft.cpp:15-58, factor2_slm_fft.cpp:16-86), re-derived for
// wave64, 160 KiB LDS and Stockham stages exchanged through LDS.
#include "../base/math.hpp"
#include "bbfft/bad_configuration.hpp"
#include "bbfft/detail/generator_impl.hpp"
#include "heuristics.hpp"
#include "tuning_table.hpp"

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <numeric>
#include <sstream>
#include <string>

namespace bbfft {

std::size_t fft1d_configuration::N_fft() const {
    bool real = type != transform_type::c2c;
    return real && N % 2 == 0 ? N / 2 : N;
}

bool fft1d_configuration::pairs_k() const { return type != transform_type::c2c && N % 2 == 1; }

std::size_t fft1d_configuration::K_columns(std::size_t K) const {
    return pairs_k() ? (K + 1) / 2 : K;
}

namespace {
std::size_t padded(std::size_t n, std::size_t pad) { return pad ? n + n / pad : n; }

bool needs_lds(fft1d_configuration const &c) {
    return c.factorization.size() > 1 || c.type != transform_type::c2c || c.direct_radix() ||
           (c.flags & (fft1d_stage_in | fft1d_stage_out));
}

/// Whether the K-columns of a side with strides {1, s_N, s_K} and n entries per transform are
/// packed, i.e. consecutive K-columns are one contiguous run of memory.
bool packed_columns(std::size_t M, std::size_t n, std::array<std::size_t, 3u> const &stride) {
    return stride[0] == 1 && stride[1] == M && stride[2] == M * n;
}
} // namespace

std::size_t fft1d_configuration::in_tile_bytes() const {
    std::size_t const rb = static_cast<std::size_t>(fp);
    std::size_t const eb = (flags & (fft1d_input_f16 | fft1d_input_bf16)) ? 4
                           : type == transform_type::r2c                  ? rb
                                                                          : 2 * rb;
    return (flags & fft1d_stage_in) ? istride[2] * Kb * (pairs_k() ? 2 : 1) * eb + 12 : 0;
}

std::size_t fft1d_configuration::out_tile_bytes() const {
    std::size_t const rb = static_cast<std::size_t>(fp);
    std::size_t const eb = type == transform_type::c2r ? rb : 2 * rb;
    return (flags & fft1d_stage_out) ? ostride[2] * Kb * (pairs_k() ? 2 : 1) * eb + 12 : 0;
}

int fft1d_configuration::direct_radix() const {
    int const r = factorization.empty()
                      ? 0
                      : *std::max_element(factorization.begin(), factorization.end());
    return is_direct_radix(r) || (flags & fft1d_direct_matrix) ? r : 0;
}

std::size_t fft1d_configuration::work_group_size() const {
    std::size_t const n = Mb * Nt * Kb;
    return (flags & fft1d_direct_matrix) ? (n + 63) / 64 * 64 : n;
}

bool fft1d_configuration::local_offsets() const {
    std::size_t const kspan = (pairs_k() ? 2 : 1) * Kb + 1;
    std::size_t const eb = 2 * static_cast<std::size_t>(fp); // largest element size
    for (auto const &s : {istride, ostride}) {
        if ((Mb + (N + 2) * s[1] + kspan * s[2]) * eb >= (std::size_t(1) << 31)) {
            return false;
        }
    }
    return true;
}

std::size_t fft1d_configuration::xcd_run() const {
    std::size_t const mg = (M + Mb - 1) / Mb;
    return mg * std::max<std::size_t>(1, 16 / mg);
}

std::size_t fft1d_configuration::lds_bytes() const {
    if (!needs_lds(*this)) {
        return 0;
    }
    std::size_t np = padded(N_fft() - 1, lds_pad) + 1;
    // the direct stage keeps its table of roots of unity in LDS
    std::size_t const table = static_cast<std::size_t>(direct_radix());
    std::size_t const eb = 2 * static_cast<std::size_t>(fp);
    std::size_t const tile = std::max({Mb * Kb * np, (in_tile_bytes() + eb - 1) / eb,
                                       (out_tile_bytes() + eb - 1) / eb});
    return (tile + table) * eb;
}

std::string fft1d_configuration::identifier() const {
    std::ostringstream oss;
    oss << "bbfft_" << (direction < 0 ? 'm' : 'p') << (direction < 0 ? -direction : direction)
        << "_M" << M << "_Mb" << Mb << "_N" << N << "_f";
    for (std::size_t i = 0; i < factorization.size(); ++i) {
        oss << (i ? "x" : "") << factorization[i];
    }
    oss << "_Nt" << Nt << "_Kb" << Kb << "_f" << static_cast<int>(fp) * 8 << '_'
        << to_string(type) << "_is" << istride[0] << '_' << istride[1] << '_' << istride[2]
        << "_os" << ostride[0] << '_' << ostride[1] << '_' << ostride[2] << "_p" << lds_pad
        << "_in" << inplace_unsupported;
    if (flags) {
        oss << "_g" << flags;
    }
    if (waves_per_eu) {
        oss << "_w" << waves_per_eu;
    }
    if (load_function) {
        oss << '_' << load_function;
    }
    if (store_function) {
        oss << '_' << store_function;
    }
    if (callback_hash) {
        oss << "_cb" << std::hex << callback_hash;
    }
    return oss.str();
}

namespace gen {

std::uint64_t callback_hash(user_module const &um) {
    if (!um) {
        return 0;
    }
    std::uint64_t h = 0xcbf29ce484222325ull;
    auto mix = [&h](unsigned char b) {
        h ^= b;
        h *= 0x100000001b3ull;
    };
    for (std::size_t i = 0; i < um.length; ++i) {
        mix(static_cast<unsigned char>(um.data[i]));
    }
    mix(static_cast<unsigned char>(um.language));
    return h ? h : 1;
}

/// Stage radices for a complex FFT of length n: one stage up to `single_max`, otherwise the
/// fewest stages whose largest radix does not exceed `radix_max` (factors closest to n^(1/L)).
std::vector<int> default_factorization(std::size_t n, std::size_t single_max,
                                       std::size_t radix_max) {
    if (n <= single_max) {
        return {static_cast<int>(n)};
    }
    for (unsigned L = 2; L <= 4; ++L) {
        auto f = factor(static_cast<unsigned>(n), L);
        // drop unit factors
        std::vector<int> g;
        for (auto v : f) {
            if (v > 1) {
                g.push_back(static_cast<int>(v));
            }
        }
        int fmax = *std::max_element(g.begin(), g.end());
        if (static_cast<std::size_t>(fmax) <= radix_max || L == 4) {
            // Largest radix first: the first stage then has the fewest butterflies, which sets
            // the work-item count, and later stages loop over more butterflies per work-item.
            std::sort(g.begin(), g.end(), std::greater<int>());
            return g;
        }
    }
    return {static_cast<int>(n)};
}

} // namespace gen

namespace {

/// Real operations of a radix-r butterfly as dft_gen emits it.
double butterfly_ops(std::size_t r) {
    if (r <= 2) {
        return r == 2 ? 4.0 : 0.0;
    }
    if (r == 4) {
        return 16.0;
    }
    std::size_t const A = r % 4 == 0 ? 4 : trial_division(static_cast<unsigned>(r)).front();
    if (A == r) {
        double const h = static_cast<double>(r / 2);
        return 4.0 * h * h + 10.0 * h;
    }
    std::size_t const B = r / A;
    return static_cast<double>(B) * butterfly_ops(A) + static_cast<double>(A) * butterfly_ops(B) +
           6.0 * static_cast<double>((A - 1) * (B - 1));
}

/// Factorisations of n, largest radix first, into radices up to 16 and primes up to the
/// register limit.
void register_factorizations(std::size_t n, std::vector<int> &cur,
                             std::vector<std::vector<int>> &out) {
    if (n == 1) {
        out.push_back(cur);
        return;
    }
    if (cur.size() == 4) {
        return;
    }
    std::size_t const hi = std::min<std::size_t>(
        n, cur.empty() ? std::size_t(fft1d_max_register_radix)
                       : static_cast<std::size_t>(cur.back()));
    for (std::size_t r = hi; r >= 2; --r) {
        if (n % r == 0 && (r <= 16 || is_prime(static_cast<unsigned>(r)))) {
            cur.push_back(static_cast<int>(r));
            register_factorizations(n / r, cur, out);
            cur.pop_back();
        }
    }
}

/**
 * Tiling of a kernel whose largest radix R (a prime) runs on the matrix cores (emit_direct_matrix):
 * M tile, K tile and work-items per transform with the least estimated time. Units of work are
 * 16 columns (m, butterfly, k) by 16 output pairs; the estimate weighs idle columns and units,
 * M tiles (not staged), resident waves and groups per CU, waves per group and columns per group.
 * Fitted to 4519 kernels of 24 lengths from 37 x 2 to 509 on MI355X (fp32 and fp64; c2c, r2c and
 * c2r; about 50 MB in and out): its choice is on average 1.8 % slower than the fastest (at most
 * 34 %). With it 8 x 509 x 8192 c2c fp32 takes 325 us instead of 960 (vector sums), 8 x 254
 * fp32 27 instead of 97, 8 x 244 c2r fp64 25 instead of 128 (registers). None is found where a
 * tile's extent needs 64-bit offsets.
 */
bool choose_direct_tiling(fft1d_configuration c, std::size_t kcols, device_info const &info,
                          bool whole_m, fft1d_tuning &out) {
    std::size_t const n = c.N_fft(), M = c.M;
    std::size_t const R = static_cast<std::size_t>(
        *std::max_element(c.factorization.begin(), c.factorization.end()));
    std::size_t const NR = n / R, h = (R - 1) / 2, KT = (h + 16) / 16;
    bool const f32 = c.fp == precision::f32;
    std::size_t const wg_max = std::min<std::size_t>(1024, info.max_work_group_size);
    // the other stages: as few as possible, radices up to 16
    if (NR > 1) {
        std::vector<std::vector<int>> facs;
        std::vector<int> cur;
        register_factorizations(NR, cur, facs);
        if (!facs.empty()) {
            auto const &f = *std::min_element(facs.begin(), facs.end(), [](auto &a, auto &b) {
                return a.size() != b.size() ? a.size() < b.size() : a.front() < b.front();
            });
            c.factorization.assign(1, static_cast<int>(R));
            c.factorization.insert(c.factorization.end(), f.begin(), f.end());
        }
    }
    c.lds_pad = 0;
    c.flags |= fft1d_direct_matrix;
    bool found = false;
    double best = 0.0;
    for (std::size_t mb : {M, std::size_t(16), std::size_t(9), std::size_t(8), std::size_t(4),
                           std::size_t(3), std::size_t(2)}) {
        if (mb > M || (mb == M ? M > 32 && !whole_m : whole_m)) {
            continue;
        }
        c.Mb = mb;
        if (mb < M) { // no staged tiles: their copies need all M columns
            c.flags &= ~unsigned(fft1d_stage_in | fft1d_stage_out);
        }
        for (std::size_t kb : {1, 2, 3, 4, 5, 6, 8, 10, 12, 16, 24, 32}) {
            for (std::size_t tk : {4, 6, 8, 12, 16, 24, 32, 48, 64}) {
                c.Kb = kb;
                c.Nt = NR * tk;
                std::size_t const wg = c.work_group_size();
                if ((kb > 1 && kb >= 2 * kcols) || wg > wg_max || !c.local_offsets() ||
                    c.lds_bytes() > info.local_memory_size) {
                    continue;
                }
                std::size_t const cols = mb * kb * NR, CT = (cols + 15) / 16, W = wg / 64;
                double cost = 0.0, held = 0.0;
                for (std::size_t k = 1; k <= std::min<std::size_t>(4, KT); ++k) {
                    std::size_t const rounds = (CT * ((KT + k - 1) / k) + W - 1) / W;
                    double const t = static_cast<double>(rounds) * (static_cast<double>(k) + 0.35);
                    if (k == 1 || t < cost) {
                        cost = t;
                        held = static_cast<double>(rounds * k);
                    }
                }
                double const regs = 60.0 + held * 16.0 * (f32 && h < 32 ? 1.0 : 2.0);
                if (regs * static_cast<double>((W + 3) / 4) > 512.0) {
                    continue;
                }
                double const waves = static_cast<double>(W);
                double const groups = std::floor(info.local_memory_size / double(c.lds_bytes()));
                double const fit = std::max(
                    waves, std::floor(4.0 * std::min(8.0, std::floor(512.0 / regs)) / waves) * waves);
                double const resident = std::min({32.0, waves * groups, fit});
                double const work = cost * waves * 16.0 / (1.35 * double(cols * KT)) *
                                    double((M + mb - 1) / mb * mb) / double(M);
                // share of the matrix instructions whose results are used: below it the sums
                // stay in vector code (5 x 331 r2c fp64, 0.43: 80 us against 71; 30 x 74 r2c fp32,
                // 0.30: 22 against 17)
                double const used = double(cols * (h + 1)) / (256.0 * waves * held);
                if (used < (R <= 61 ? 0.35 : f32 ? 0.2 : 0.55) && kcols > 64) {
                    continue;
                }
                double const score = 0.414 * std::log(work) * std::min(1.0, double(h) / 40.0) +
                                     0.177 / resident + (mb < M ? 0.056 : 0.0) -
                                     0.0788 * std::log2(waves) +
                                     0.221 * std::min(2.0, 1.0 / groups) +
                                     0.1024 * std::log2(double(cols) / 16.0);
                if (!found || score < best) {
                    found = true;
                    best = score;
                    out.factorization = c.factorization;
                    out.Nt = c.Nt;
                    out.Mb = mb;
                    out.Kb = kb;
                    out.lds_pad = 0;
                    out.no_pad = true;
                }
            }
        }
    }
    return found;
}

/// Work-items of a launch with whole waves (all M columns in a tile).
std::size_t work_items(std::size_t M, fft1d_tuning const &t, std::size_t kcols) {
    return (kcols + t.Kb - 1) / t.Kb * ((M * t.Nt * t.Kb + 63) / 64 * 64);
}

/**
 * Tiling of a kernel that holds all M columns of Kb transforms in one work-group (staged tiles):
 * the factorisation, work-items per transform and K tile with the least estimated time. The
 * estimate is linear in what separated the candidates of a sweep on MI355X (f32 and f64; c2c,
 * r2c and c2r; 28 shapes from 1 x 16 to 17 x 363; about 100 MB in and out; 3432 kernels):
 * vector operations per element with idle lanes counted, stages, resident waves per CU (from
 * LDS, registers and the number of work-groups), waves per group (barriers), registers per
 * work-item and lines shared by neighbouring tiles. Its choice is on average 1.6 % slower than
 * the fastest candidate (at most 18 %); the fewest-stages tiling with about 256 work-items per
 * group is 7 % slower for c2c and, without staged tiles, 32 % over all types.
 */
bool choose_tiling(fft1d_configuration c, std::size_t kcols, device_info const &info,
                   fft1d_tuning &out) {
    std::size_t const n = c.N_fft(), M = c.M;
    std::vector<std::vector<int>> facs;
    if (n == 1) {
        facs.push_back({1});
    } else {
        std::vector<int> cur;
        register_factorizations(n, cur, facs);
    }
    std::size_t stages = 4;
    for (auto const &f : facs) {
        stages = std::min(stages, f.size());
    }
    std::size_t const wg_max = std::min<std::size_t>(1024, info.max_work_group_size);
    double const real = c.type != transform_type::c2c ? 1.0 : 0.0;
    double const words = c.fp == precision::f32 ? 2.0 : 4.0; // registers of a complex value
    c.lds_pad = n >= 32 && (stages > 1 || real > 0.0) ? 16 : 0;
    // Stages beyond the fewest. A stage more is a rounding more, which fp64 results show (96 c2c
    // 1.63e-16 against 1.53e-16, 384 c2c 2.01e-16 / 1.97e-16, 12 r2c 1.38e-16 / 1.22e-16) and which
    // only some shapes are faster for (c2c 96 to 300: 0.9 to 1.03 of the time; 384 and 500 with four
    // stages 1.02 to 1.1; r2c and c2r of 256 to 512 with three 0.8 to 0.95). Half-precision input,
    // whose tiles are read element by element, pays for it (1 x 100 x 10000 f16 6.1 us against 5.0).
    bool const half_in = (c.flags & (fft1d_input_f16 | fft1d_input_bf16)) != 0;
    if (c.fp == precision::f32 && !half_in) {
        ++stages;
    } else if (stages == 1 ? n >= 8 : stages == 2 && !half_in && (real > 0.0 || n >= 256)) {
        ++stages;
    }
    bool found = false;
    double best = 0.0;
    c.Mb = M;
    for (auto const &f : facs) {
        if (f.size() > stages) {
            continue;
        }
        c.factorization = f;
        for (std::size_t which = 0; which < std::min<std::size_t>(2, f.size()); ++which) {
            std::size_t const Nt = n / static_cast<std::size_t>(f[which]);
            // A wide prime radix spread over as many work-items as the other stage has points leaves
            // most of them idle (4 x 58 c2c fp32 8.7 us, 6.6 with one butterfly each), which the
            // estimate, fitted to radices up to 17, sees too little of.
            if ((which && (f[1] == f[0] || f[0] > 23)) || M * Nt > wg_max) {
                continue;
            }
            c.Nt = Nt;
            double ops = 0.0, held = 0.0; // per work-item: operations, complex values in registers
            for (std::size_t s = 0; s < f.size(); ++s) {
                std::size_t const r = static_cast<std::size_t>(f[s]);
                double const rounds = static_cast<double>((n / r + Nt - 1) / Nt);
                double const R = static_cast<double>(r);
                ops += rounds * (butterfly_ops(r) + (s ? 6.0 * (R - 1.0) : 0.0) + 4.0 * R);
                held = std::max(held, rounds * R);
            }
            for (std::size_t items : {64u, 96u, 128u, 192u, 256u}) {
                c.Kb = std::min(kcols, std::max<std::size_t>(1, items / (M * Nt)));
                std::size_t const wg = c.work_group_size();
                if (c.lds_bytes() > info.local_memory_size || wg > wg_max) {
                    continue;
                }
                double const waves = static_cast<double>((wg + 63) / 64);
                double const regs = 36.0 + words * held;
                // A group of many waves caps the registers of each: 22 x 205 c2c fp64 (41 x 5) with
                // 902 work-items spilled, 162 us against 24.
                if (4.0 * std::floor(512.0 / regs) < waves) {
                    continue;
                }
                double const groups = static_cast<double>((kcols + c.Kb - 1) / c.Kb);
                double resident = std::floor(info.local_memory_size / double(c.lds_bytes())) * waves;
                resident = std::min(resident, waves * groups / 256.0);
                resident = std::min(
                    resident,
                    waves * std::max(1.0, std::floor(4.0 * std::min(8.0, std::floor(512.0 / regs)) /
                                                     waves)));
                resident = std::min(resident, 32.0);
                double const per_element =
                    ops * waves * 64.0 / static_cast<double>(n * M * c.Kb);
                // lines that a tile shares with its neighbours (they move twice)
                double edges = 0.0;
                for (std::size_t b : {c.in_tile_bytes(), c.out_tile_bytes()}) {
                    if (b && (b - 12) % 128 != 0) {
                        edges += 128.0 / static_cast<double>(b);
                    }
                }
                double const score =
                    1.2e-3 * per_element + 4.6e-2 * static_cast<double>(f.size()) +
                    1.13 / resident + 4.8e-3 * std::log2(waves) + 2.2e-3 * words * held +
                    0.48 * edges;
                if (!found || score < best) {
                    found = true;
                    best = score;
                    out.factorization = f;
                    out.Nt = Nt;
                    out.Mb = M;
                    out.Kb = c.Kb;
                    out.lds_pad = c.lds_pad;
                    out.no_pad = c.lds_pad == 0;
                }
            }
        }
    }
    return found;
}

} // namespace

fft1d_configuration configure_fft1d(configuration const &cfg, device_info const &info,
                                    fft1d_tuning const &tuning_in, unsigned variant) {
    if (cfg.dim != 1) {
        throw bad_configuration("configure_fft1d requires a 1-D configuration");
    }
    if (cfg.istride[0] != 1 || cfg.ostride[0] != 1) {
        throw bad_configuration("Stride s_0 != 1 is not supported");
    }
    if ((cfg.type == transform_type::r2c && cfg.dir != direction::forward) ||
        (cfg.type == transform_type::c2r && cfg.dir != direction::backward)) {
        throw bad_configuration("r2c must be forward and c2r must be backward");
    }
    std::size_t const M = cfg.shape[0], N = cfg.shape[1], K = cfg.shape[2];
    if (M == 0 || N == 0 || K == 0) {
        throw bad_configuration("Tensor shape must not contain zeros");
    }
    // Without explicit tuning, a measured entry of the persisted table (if any) is used; its
    // K tile is clamped to the number of K columns below.
    fft1d_tuning tuning = tuning_in;
    bool const explicit_tuning = !tuning_in.factorization.empty() || tuning_in.Nt ||
                                 tuning_in.Mb || tuning_in.Kb || tuning_in.lds_pad ||
                                 tuning_in.no_pad || tuning_in.has_flags;
    unsigned const all_flags =
        ((tuning_in.has_flags ? tuning_in.flags : 0u) | variant) & ~unsigned(fft1d_access_by_rule);
    bool const half_in = (all_flags & (fft1d_input_f16 | fft1d_input_bf16)) != 0;
    bool const mfma = (all_flags & fft1d_mfma) != 0;
    std::size_t const half = N / 2 + 1;
    bool const in = packed_columns(M, cfg.type == transform_type::c2r ? half : N,
                                   {cfg.istride[0], cfg.istride[1], cfg.istride[2]});
    bool const outp = packed_columns(M, cfg.type == transform_type::r2c ? half : N,
                                     {cfg.ostride[0], cfg.ostride[1], cfg.ostride[2]});
    if (!explicit_tuning && info.type == device_type::gpu && info.max_subgroup_size() == 64) {
        gen::lookup_tuning(cfg.fp, cfg.type, N, M, all_flags, tuning, in || outp);
        if (char const *m = std::getenv("BBFFT_TABLE_FLAGS_CLEAR")) { // A/B: drop entry flags
            tuning.flags &= ~static_cast<unsigned>(std::strtoul(m, nullptr, 0));
        }
        // The table is measured on plain kernels; the load-first tile loop needs direct global
        // loads, so a plan with callbacks keeps the entry's tiling without it, and without the
        // entry's occupancy target and persistent grid: the callback's code adds registers (a
        // filter-multiplying load callback on the 128-point pass of 32 x 128^3 spilled 46
        // VGPRs at 4 waves per SIMD and needs 146 without the cap, no spills).
        if (cfg.callbacks) {
            tuning.flags &= ~static_cast<unsigned>(fft1d_prefetch);
            tuning.waves_per_eu = 0;
            tuning.groups_per_cu = 0;
            if (char const *w = std::getenv("BBFFT_CALLBACK_WAVES")) { // A/B
                tuning.waves_per_eu = static_cast<unsigned>(std::atoi(w));
            }
            // A kernel with a load callback streams its stores past the last-level cache: the
            // callback may read side data (a filter read once per batch) that the kernel's
            // output would otherwise evict. BBFFT_CALLBACK_NT=off keeps the entry's stores.
            char const *nt = std::getenv("BBFFT_CALLBACK_NT");
            if (cfg.callbacks.load_function && tuning.has_flags &&
                !(nt && std::string(nt) == "off")) {
                tuning.flags &= ~unsigned(fft1d_access_by_rule);
                tuning.flags |= fft1d_nontemporal_store;
            }
        }
    }
    // Access flags by rule, of a whole tiling; any other entry's or caller's flags apply as given.
    bool const by_rule = tuning.has_flags && (tuning.flags & fft1d_access_by_rule) &&
                         !tuning.factorization.empty() && tuning.Nt && tuning.Mb && tuning.Kb;
    bool const given_flags = tuning.has_flags && !(tuning.flags & fft1d_access_by_rule);
    bool const streamed = by_rule && (tuning.flags & fft1d_nontemporal_load);
    if (tuning.flags & fft1d_access_by_rule) {
        variant |= all_flags & (fft1d_input_f16 | fft1d_input_bf16 | fft1d_mfma);
        tuning.flags &= half_in ? 0u : unsigned(fft1d_direct_matrix); // a property of the tiling
        tuning.has_flags = tuning.flags != 0;
    }

    fft1d_configuration c = {};
    c.direction = static_cast<int>(cfg.dir);
    c.M = M;
    c.N = N;
    c.fp = cfg.fp;
    c.type = cfg.type;
    c.istride = {cfg.istride[0], cfg.istride[1], cfg.istride[2]};
    c.ostride = {cfg.ostride[0], cfg.ostride[1], cfg.ostride[2]};
    c.load_function = cfg.callbacks.load_function;
    c.store_function = cfg.callbacks.store_function;
    c.callback_hash = gen::callback_hash(cfg.callbacks);
    std::size_t const nfft = c.N_fft();
    std::size_t const kcols = c.K_columns(K);

    bool inplace_refused = false;
    bool const real = cfg.type != transform_type::c2c;
    std::size_t const eb = 2 * static_cast<std::size_t>(cfg.fp);
    // Staged tiles are addressed by 32-bit offsets. `Kb` 0: the tile's K-columns are not chosen
    // yet (at most 256).
    auto const stageable = [&](std::size_t Kb) {
        fft1d_configuration t = c;
        t.Mb = M;
        t.Kb = Kb ? Kb : 256;
        return (in || outp) && t.local_offsets();
    };
    // Adds the flags of a kernel whose packed sides may be staged; `items`: work-items of the
    // launch.
    auto const stage = [&](std::size_t items) {
        tuning.flags |= fft1d_per_tile_ids;
        std::size_t const half_eb = half_in ? 4 : eb;
        std::size_t const bytes =
            M * K *
            ((cfg.type == transform_type::r2c ? N * eb / 2
                                              : (cfg.type == transform_type::c2r ? half : N) * half_eb) +
             (cfg.type == transform_type::c2r ? N * eb / 2
                                              : (cfg.type == transform_type::r2c ? half : N) * eb));
        auto const &f = tuning.factorization;
        int const r = f.empty() ? 0 : *std::max_element(f.begin(), f.end());
        if (r <= 32 && bytes <= (real ? 26u : 34u) << 20) {
            // Data that fits the 32 MB of L2: plain loads find what the last kernel left there,
            // and streamed stores take the write-back off the kernel's end. The copies' barriers
            // have nothing to win back, except in real transforms of short rows. To the spectrum
            // and back in microseconds, in a replayed graph (copies / plain / plain with streamed
            // stores): 1 x 64 x 16384 fp32 8.0 / 7.5 / 6.8, 1 x 100 x 5242 fp64 9.4 / 8.5 / 7.8,
            // 8 x 64 x 4096 fp32 10.7 / 13.6 / 10.4, 1 x 64 x 32768 10.9 / 14.4 / 11.6; 8 x 64 x
            // 8192 23.3 / 23.1 / 24.0. r2c 8 x 64 x 4096 10.4 / 9.6 / 8.7, 1 x 64 x 32768 11.9 /
            // 11.7 / 11.0 (10.5: copies, plain loads).
            if (!c.store_function && (outp || M * eb >= 24)) {
                tuning.flags |= fft1d_nontemporal_store;
            }
            if (real && M * eb < 40 && N < 256) {
                tuning.flags |= (in && !c.load_function ? fft1d_stage_in : 0u) |
                                (outp && !c.store_function ? fft1d_stage_out : 0u);
            }
            tuning.has_flags = true;
            return;
        }
        // The copies add two barriers to a work-group's latency: below 8 waves per CU there is too
        // little else to hide it.
        bool const filled = items >= 8 * 64 * 256;
        if (in && !c.load_function && filled) {
            // Streamed loads leave nothing of the input in the 256 MB last-level cache. Where input
            // and output fit there, plain ones find what the last kernel or call left: repeated
            // calls (plain / streamed, geometric means over 17 shapes, M 1 to 17) of 38 MB c2c 0.84,
            // 50 MB 0.93, 70 to 220 MB 0.90 to 0.92, r2c and c2r 0.84 to 0.96; from memory 1.01 to
            // 1.03. (540 MB 0.91 and 1.05, 640 MB 1.07 and 1.05.) A row may stream all the same.
            tuning.flags |= fft1d_stage_in;
            if (streamed || bytes > std::size_t(256) << 20) {
                tuning.flags |= fft1d_nontemporal_load;
            }
        }
        if (!c.store_function && (outp || M * eb >= 24) && filled) {
            tuning.flags |= (outp ? fft1d_stage_out : 0u) | fft1d_nontemporal_store;
        }
        if (!filled && r <= 32 && M * eb >= 24) { // 15 x 58 x 1607 c2c fp64 12.3 us, plain 14.9
            tuning.flags |= fft1d_nontemporal_load | fft1d_nontemporal_store;
        }
        tuning.has_flags = true;
        c.Mb = M;
        c.Kb = tuning.Kb;
        c.flags = tuning.flags;
        // shared lines: 5 x 315 x 15000 c2r fp32 39.7 us against 43.4, 1 x 512 r2c 49.7 / 50.5
        if (tuning.Kb && ((c.in_tile_bytes() && (c.in_tile_bytes() - 12) % 128 != 0) ||
                          (c.out_tile_bytes() && (c.out_tile_bytes() - 12) % 128 != 0))) {
            tuning.flags |= fft1d_xcd_runs;
        }
        c.flags = 0;
    };
    if (by_rule && tuning.Mb >= M && !mfma && !half_in && info.type == device_type::gpu) {
        // The tiling of a staged kernel, where the layout allows one: 8 x 16 c2c fp32 166 us (524288
        // K-columns) against 192 (load-first loop), 8 x 512 176 / 183, 8 x 384 c2r 181 / 233. Its
        // persistent grid, if any, is for launches that give each work-group 32 tiles or more (8 x
        // 512 fp64: 32768 K-columns 694 us against 711 staged, 8192 182 / 182, 1000 26.4 / 24.6).
        std::size_t const columns = std::size_t(32) * 256 * tuning.groups_per_cu * tuning.Kb;
        if (!stageable(tuning.Kb) || tuning_in.unstaged) {
            tuning.has_flags = tuning.flags || tuning.groups_per_cu; // else the default hints
        } else if (columns && kcols >= columns) {
            tuning.flags |= fft1d_per_tile_ids;
            tuning.has_flags = true;
        } else {
            tuning.groups_per_cu = 0;
            stage(work_items(M, tuning, kcols));
        }
    }
    // Shapes without a table entry: when the K-columns of a side are packed, all M columns of a
    // tile sit in LDS and that side moves in 16-byte pieces, streamed past the caches.
    if (!explicit_tuning && tuning.factorization.empty() && info.type == device_type::gpu &&
        !mfma && !tuning_in.unstaged) {
        auto const f = gen::default_factorization(nfft, 16, 16);
        std::size_t const r = static_cast<std::size_t>(*std::max_element(f.begin(), f.end()));
        bool const registers = r <= static_cast<std::size_t>(fft1d_max_register_radix);
        std::size_t const Nt = nfft / r;
        // c2c fp32 with M = 2 or 3 keeps the fewest-stages tiling, staged: its factors, tile and
        // padding are a fixed part of the heuristic's interface (the estimate's choice is 1-9 %
        // faster there)
        bool const keep = !real && cfg.fp == precision::f32 && !half_in && (M == 2 || M == 3) &&
                          r <= 16 && M * Nt <= 512;
        fft1d_tuning const untiled = tuning;
        // Large prime factors on the matrix cores (not with half-precision input, whose access
        // flags have no such kernel: 4 x 37 x 110000 f16 had the tiling of matrix sums without
        // them, 234 us against 139). Radices up to 64 also run in registers, which
        // stays the faster way for fp32 below 37 (31 x 2 and 31 x 4, 8 columns: equal), for fp64
        // below 31, and for M tiles up to 61 in fp32 and 41 in fp64 (30 columns: 53 x 2 fp32 36 us
        // against 44, 37 x 2 fp64 29 against 35; but 53 x 2 fp64 88 against 38).
        int const large = cfg.fp == precision::f32 ? 37 : 31;
        bool matrix = !half_in && static_cast<int>(r) >= large &&
                      is_prime(static_cast<unsigned>(r)) &&
                      std::count(f.begin(), f.end(), static_cast<int>(r)) == 1;
        c.factorization = f;
        c.Nt = Nt;
        if (!registers) { // the direct stage in vector code, which also fixes in-place use below
            std::size_t const units = (r - 1) / 2 + 1, per_item = cfg.fp == precision::f32 ? 8 : 6;
            c.Nt = nfft / r * ((units + per_item - 1) / per_item);
        }
        c.Mb = M;
        c.Kb = 1;
        c.lds_pad = nfft >= 32 && (f.size() > 1 || real) ? 16 : 0;
        c.flags = 0;
        // Real transforms run in place when one tile holds all M columns: up to 64 columns, 512
        // work-items and 64 KB of LDS for a single K-column.
        bool const whole_m =
            M <= std::max<std::size_t>(1, std::min<std::size_t>(64, 512 / c.Nt)) &&
            (M == 1 || c.lds_bytes() <= 64 * 1024);
        inplace_refused = real && !whole_m;
        c.flags = all_flags | (in ? fft1d_stage_in : 0u) | (outp ? fft1d_stage_out : 0u);
        matrix = matrix && choose_direct_tiling(c, kcols, info, real && whole_m, tuning) &&
                 (tuning.Mb == M || r > (cfg.fp == precision::f32 ? 61 : 41));
        if (!matrix) {
            tuning = untiled;
        }
        bool staged = matrix ? (in || outp) && tuning.Mb == M
                             : (in || outp) && (keep || choose_tiling(c, kcols, info, tuning));
        // Tiles of 36 KB and more leave a CU four groups, too few to overlap the copies of one with
        // the stages of the others: c2c whose default tile holds all M columns keeps that tile and
        // its streamed accesses. fp64, 256 MB / 64 MB in and out, staged against that: 9 x 256 50.0 /
        // 16.0 us, 46.9 / 14.5; 12 x 220 57.0 / 19.0, 51.0 / 15.5; 14 x 243 70.2 / 21.2, 58.5 /
        // 17.8; fp32 48 x 128 49.8 / 15.4, 47.1 / 12.5. (Default M tiles lose to staged tiles of any
        // size: 12 x 384 fp64 108 us, staged 66.)
        bool const large_tile = !real && !half_in && whole_m && M * N * eb >= 36000;
        if (staged && !matrix && (large_tile || !stageable(tuning.Kb))) {
            tuning = untiled;
            staged = false;
        }
        if (staged && !matrix && !keep && !(real && whole_m)) {
            // Tiles above half the LDS leave a CU with nothing to overlap a tile's copies, and
            // tiles of all M columns of few K-columns leave CUs idle: the tiles of layouts that
            // are not packed instead (real transforms that run in place keep all M columns; 36 x
            // 243 r2c fp32, 4 K-columns, 5.2 us against 6.1 staged).
            fft1d_configuration t = c;
            t.factorization = tuning.factorization;
            t.Kb = tuning.Kb;
            t.lds_pad = tuning.lds_pad;
            t.flags = 0;
            staged = t.lds_bytes() <= info.local_memory_size / 2 &&
                     (real ? kcols >= 64 : M == 1 || kcols >= 256 || M * Nt <= 64);
            if (!staged) {
                tuning = untiled;
            }
        }
        if (matrix) {
            tuning.flags = fft1d_per_tile_ids | fft1d_direct_matrix;
        }
        // rows of whole 64-byte segments on both sides
        std::size_t const seg = 64 / static_cast<std::size_t>(cfg.fp);
        bool const aligned = M % seg == 0 && c.istride[1] % seg == 0 && c.ostride[1] % seg == 0 &&
                             c.istride[2] % seg == 0 && c.ostride[2] % seg == 0;
        if (staged) {
            stage(keep ? M * Nt * kcols : work_items(M, tuning, kcols));
        } else if (matrix) {
            tuning.flags |= fft1d_xcd_runs;
            tuning.has_flags = true;
        } else if (registers && !whole_m && !(real && (aligned || kcols * ((M + 63) / 64) < 64))) {
            // M tiles, where the default tile does not hold all M columns (where it does, its
            // streamed accesses are the faster ones: 6 x 363 c2c fp64, padded rows, 206 us against
            // 225, 16 x 128 fp32 11.9 / 14.3; halved for few K-columns, 5 x 500 fp64 x 209 packed
            // 9.8 us against 5.8). Rows of whole 128-byte lines are stored past the caches, 128 to
            // 256 bytes per tile: 4704 x 80 x 16 fp32 20.0 us (32 columns; 25.1 with 64 columns and
            // hoisted ids, 21.5 with plain stores). Streamed loads as well: 19.4, but data that the
            // last kernel left in a cache is lost (512 x 64 x 64 to the spectrum and back 13.2
            // against 10.5; 8320 x 128 x 32 from HBM 95.6 against 86.6). Otherwise neighbouring M
            // tiles share the lines at their seams: the widest tiles, plain accesses and neighbours
            // on one XCD; 17 x 512 x 2757 fp32 81 us (9 columns) against 323 (6 columns streamed,
            // neighbours on different XCDs) and 130 (9 columns plain, different XCDs).
            std::size_t const line = 128 / eb;
            bool const lines = M % line == 0 && c.istride[1] % line == 0 &&
                               c.ostride[1] % line == 0 && c.istride[2] % line == 0 &&
                               c.ostride[2] % line == 0 && !real;
            tuning.factorization = f;
            tuning.Nt = Nt;
            std::size_t mb = std::min<std::size_t>(64, std::max<std::size_t>(1, 1024 / Nt));
            if (lines) {
                mb = std::max(line, std::min(2 * line, 512 / Nt));
            }
            // few K-columns: smaller tiles, of whole 64-byte segments where rows consist of them,
            // until there is a work-group for every other CU or a tile is one wave (41 x 220 c2c
            // fp32 x 76, two tiles 7.4 us, four 8.8)
            std::size_t const few = std::max<std::size_t>(1, 64 / Nt), part = 64 / eb;
            std::size_t const parts = (128 + kcols - 1) / kcols;
            if (!real && kcols * ((M + mb - 1) / mb) < 128) {
                mb = std::min(mb, std::max(few, (M + parts - 1) / parts));
                if (M % part == 0 && mb > part) {
                    mb -= mb % part;
                }
            }
            std::size_t mg = (M + mb - 1) / mb;
            c.factorization = f;
            c.Nt = Nt;
            c.Kb = 1;
            c.flags = 0;
            c.lds_pad = nfft >= 32 && (f.size() > 1 || real) ? 16 : 0;
            for (c.Mb = (M + mg - 1) / mg;
                 c.Mb > 1 && (c.lds_bytes() > info.local_memory_size / 2 || c.Mb * Nt > 1024);) {
                ++mg;
                c.Mb = (M + mg - 1) / mg;
            }
            tuning.Mb = c.Mb;
            if (!real && kcols < 256) {
                tuning.Kb = 1;
            }
            tuning.lds_pad = c.lds_pad;
            tuning.no_pad = c.lds_pad == 0;
            tuning.flags = fft1d_per_tile_ids;
            if (lines && c.Mb % line == 0) {
                tuning.flags |= fft1d_nontemporal_store;
            } else if (M * Nt * kcols >= 8 * 64 * 256) {
                tuning.flags |= fft1d_xcd_runs;
            }
            tuning.has_flags = true;
        }
        c.flags = 0;
    }

    if (half_in) {
        if ((all_flags & fft1d_input_f16) && (all_flags & fft1d_input_bf16)) {
            throw bad_configuration("Choose one half-precision input format");
        }
        if (cfg.type != transform_type::c2c || cfg.fp != precision::f32) {
            throw bad_configuration("Half-precision input requires a c2c fp32 transform");
        }
        if (cfg.callbacks) {
            throw bad_configuration("Half-precision input does not support callbacks");
        }
    }
    if (mfma) {
        if (!half_in) {
            throw bad_configuration("The MFMA stage requires half-precision input");
        }
        if (nfft % 16 != 0 || nfft < 32) {
            throw bad_configuration("The MFMA stage requires N divisible by 16 and N >= 32");
        }
        if (!tuning.factorization.empty() && tuning.factorization[0] != 16) {
            throw bad_configuration("The MFMA stage requires a first radix of 16");
        }
    }
    if (!tuning.factorization.empty()) {
        std::size_t p = 1;
        for (auto f : tuning.factorization) {
            if (f < 1) {
                throw bad_configuration("factorization entries must be positive");
            }
            p *= static_cast<std::size_t>(f);
        }
        if (p != nfft) {
            throw bad_configuration("factorization does not multiply to the FFT length");
        }
        c.factorization = tuning.factorization;
    } else {
        // Radices up to 16: a larger radix means more elements per work-item (registers) and
        // fewer work-items per transform. On MI355X the 2-stage radix-20..32 splits of N = 243,
        // 384, 500, 512 at M <= 4 reached 3.1-5.8 TB/s against 5.7-6.6 TB/s with radix <= 16.
        std::size_t const single_max = 16;
        std::size_t const radix_max = 16;
        c.factorization = gen::default_factorization(nfft, single_max, radix_max);
        if (mfma) {
            c.factorization = gen::default_factorization(nfft / 16, 16, 16);
            c.factorization.insert(c.factorization.begin(), 16);
        }
    }
    // Radices above the register limit run as a direct DFT stage (one per kernel, odd radix:
    // the symmetric-pair sums need no self-paired index), as the reference falls back to
    // basic_esum for prime factors above its register budget.
    int direct = 0;
    for (auto f : c.factorization) {
        if (is_direct_radix(f)) {
            if (f % 2 == 0) {
                throw bad_configuration("Radix " + std::to_string(f) +
                                        " exceeds the in-register limit (" +
                                        std::to_string(fft1d_max_register_radix) +
                                        ") and is even; split it into smaller radices");
            }
            if (direct) {
                throw bad_configuration("N = " + std::to_string(N) +
                                        " has two factors above the in-register limit (" +
                                        std::to_string(fft1d_max_register_radix) +
                                        "); at most one is supported");
            }
            direct = f;
        }
    }
    if (direct && mfma) {
        throw bad_configuration("The MFMA stage does not combine with a direct DFT stage");
    }
    if (tuning.has_flags && (tuning.flags & fft1d_direct_matrix)) {
        int const r = *std::max_element(c.factorization.begin(), c.factorization.end());
        if (r < 17 || !is_prime(static_cast<unsigned>(r)) ||
            std::count(c.factorization.begin(), c.factorization.end(), r) != 1) {
            throw bad_configuration("Matrix sums need one prime radix above 16 as the largest");
        }
        direct = r;
    }
    // The MFMA stage does not use the work-items-per-transform split; later stages set it.
    int const rmax = mfma ? *std::max_element(c.factorization.begin() + 1, c.factorization.end())
                          : *std::max_element(c.factorization.begin(), c.factorization.end());
    if (direct) {
        // Work-item t of a transform serves butterfly t % (N_fft / R) of the direct stage and
        // output pairs t / (N_fft / R) + b Tk of it; Tk is chosen so that each work-item keeps
        // about 8 (fp32) or 6 (fp64) output pairs in registers.
        std::size_t const NRd = nfft / static_cast<std::size_t>(direct);
        std::size_t const units = static_cast<std::size_t>(direct - 1) / 2 + 1;
        std::size_t const per_item = cfg.fp == precision::f32 ? 8 : 6;
        std::size_t const Tk = (units + per_item - 1) / per_item;
        c.Nt = tuning.Nt ? tuning.Nt : NRd * Tk;
        if (c.Nt % NRd != 0) {
            throw bad_configuration("With a direct DFT stage of radix " + std::to_string(direct) +
                                    " the work-items per transform must be a multiple of " +
                                    std::to_string(NRd));
        }
    } else {
        c.Nt = tuning.Nt ? tuning.Nt : nfft / static_cast<std::size_t>(rmax);
    }

    std::size_t const wg_max = std::min<std::size_t>(1024, info.max_work_group_size);
    if (c.Nt == 0 || c.Nt > wg_max) {
        throw bad_configuration("Invalid number of work-items per transform");
    }
    if (tuning.Mb) {
        c.Mb = std::min(tuning.Mb, M);
    } else {
        std::size_t mmax = std::max<std::size_t>(1, std::min<std::size_t>(64, 512 / c.Nt));
        std::size_t mg = (M + mmax - 1) / mmax;
        c.Mb = (M + mg - 1) / mg;
    }
    if (c.Mb * c.Nt > wg_max) {
        throw bad_configuration("M tile times work-items per transform exceeds work-group size");
    }

    c.lds_pad = 0;
    if (tuning.lds_pad) {
        c.lds_pad = tuning.lds_pad;
    } else if (!tuning.no_pad && (c.factorization.size() > 1 || cfg.type != transform_type::c2c)) {
        c.lds_pad = nfft >= 32 ? 16 : 0;
    }
    if (c.lds_pad & (c.lds_pad - 1)) {
        throw bad_configuration("lds_pad must be a power of two");
    }

    std::size_t const lds_limit = std::min<std::size_t>(info.local_memory_size, 64 * 1024);
    if (!tuning.Mb) {
        // Shrink the M tile until one K-column tile fits the LDS budget.
        c.Kb = 1;
        std::size_t mg = (M + c.Mb - 1) / c.Mb;
        while (c.Mb > 1 && c.lds_bytes() > lds_limit) {
            ++mg;
            c.Mb = (M + mg - 1) / mg;
        }
    }
    if (tuning.Kb && (tuning.flags & fft1d_direct_matrix)) {
        c.Kb = tuning.Kb; // whole waves: K-columns beyond kcols are idle
    } else if (tuning.Kb) {
        c.Kb = std::min(tuning.Kb, kcols);
    } else {
        std::size_t target = 256;
        std::size_t kb = std::max<std::size_t>(1, target / (c.Mb * c.Nt));
        kb = std::min(kb, kcols);
        c.Kb = kb;
        while (c.Kb > 1 && c.lds_bytes() > lds_limit) {
            --c.Kb;
        }
    }
    if (mfma) {
        // Matrix instructions read all 64 lanes of a wave: whole waves only (the extra K
        // columns are inactive when K is smaller).
        std::size_t const step = 64 / std::gcd<std::size_t>(c.Mb * c.Nt, 64);
        c.Kb = (c.Kb + step - 1) / step * step;
        if (c.lds_bytes() > lds_limit) {
            throw bad_configuration("MFMA kernel tile exceeds the LDS budget");
        }
    }
    if (c.work_group_size() > wg_max) {
        throw bad_configuration("Work-group size exceeds the device limit");
    }
    if (c.lds_bytes() > info.local_memory_size) {
        throw bad_configuration("Work-group exceeds the local memory size");
    }
    // Access hints without a measured entry: streaming (non-temporal) loads and stores when a
    // work-group's M run is at least 24 contiguous bytes. Measured on MI355X for untuned shapes
    // (heuristic tiling, about 1 GB per buffer, flags 0 vs 3): fp32 M=4 N=500 +11 %, M=3
    // N=384 +8 %, M=4 N=128 +2 %, M=16 N=64 +4 %, fp64 M=2 N=500 +5 %; fp32 M=1 N=60 -55 %,
    // M=1 N=100 -16 %, M=2 N=243 -13 %, r2c M=1 N=500 -18 %, c2r M=2 N=243 -6 %.
    unsigned default_hints = 0;
    if (info.type == device_type::gpu &&
        c.Mb * 2 * static_cast<std::size_t>(c.fp) >= 24) {
        default_hints = fft1d_nontemporal_load | fft1d_nontemporal_store;
    }
    c.flags = (tuning.has_flags ? tuning.flags : default_hints) | variant;
    // Lengths whose sums run in vector code keep streaming small data: 8 x 509 x 258 f16 79 us
    // against 86 (x 2000 243 / 210).
    bool const small_sums = direct && M * N * K * (4 + eb) <= std::size_t(34) << 20;
    if (half_in && !given_flags && (!explicit_tuning || by_rule) && !small_sums &&
        info.type == device_type::gpu && c.Mb == M) {
        // Half-precision input: four bytes per element leave the loads cheap and their lines
        // shared by neighbouring accesses, so they go through the caches, element by element.
        // MI355X, vector kernels, streamed loads before: 8 x 64 x 60000 62 -> 54 us, 16 x 384 x 3000
        // 65 -> 43. The output is staged beyond the 32 MB of L2 where rows are shorter than 32
        // bytes (3 x 61 f16 204 us direct, 148 staged). Longer rows gain from 0.9 GB on (4 x 512 x
        // 32768 130 / 135, x 131072 523 / 512, with two K-columns a tile, a single wave having
        // nothing to overlap its copies: 531 with one), radices above 32 not at all (16 x 122 491 /
        // 577); on the matrix cores, whose tiles take more of a CU, long transforms beyond 1 GB (4
        // x 512 x 40000 163 / 162, x 98304 405 / 390; 2 x 256 x 240000 241 / 248).
        c.flags = variant | fft1d_per_tile_ids;
        if (outp || M * eb >= 24) {
            c.flags |= fft1d_nontemporal_store;
        }
        std::size_t const bytes = M * N * K * (4 + eb);
        bool const staged = mfma           ? N >= 512 && bytes > std::size_t(1) << 30
                            : M * eb < 32 ? bytes > std::size_t(34) << 20
                                           : rmax <= 32 && bytes > std::size_t(900) << 20;
        if (outp && staged) {
            fft1d_configuration const plain = c;
            c.flags |= fft1d_stage_out | fft1d_xcd_runs;
            if (!mfma && c.Mb * c.Nt * c.Kb <= 64) {
                c.Kb = std::min(2 * c.Kb, kcols);
            }
            if (c.lds_bytes() > info.local_memory_size || !c.local_offsets()) {
                c = plain;
            }
        }
    }
    if (tuning.waves_per_eu > 8) {
        throw bad_configuration("waves_per_eu must be 0..8");
    }
    c.waves_per_eu = tuning.waves_per_eu;
    c.groups_per_cu = tuning.groups_per_cu;
    if (c.flags & fft1d_prefetch) {
        if (cfg.type == transform_type::c2r || cfg.callbacks || (c.flags & fft1d_mfma) ||
            direct || (c.flags & fft1d_per_tile_ids)) {
            throw bad_configuration("Tile prefetching requires a c2c or r2c kernel without "
                                    "callbacks, MFMA, direct DFT stage or per-tile ids");
        }
    }
    if (c.flags & (fft1d_stage_in | fft1d_stage_out)) {
        std::size_t const half = cfg.shape[1] / 2 + 1;
        std::size_t const n_in = cfg.type == transform_type::c2r ? half : N;
        std::size_t const n_out = cfg.type == transform_type::r2c ? half : N;
        if ((c.flags & fft1d_stage_in) &&
            (c.Mb != M || !packed_columns(M, n_in, c.istride) || c.load_function || mfma ||
             (c.flags & fft1d_prefetch))) {
            throw bad_configuration("Staged input needs packed columns, one M tile, no load "
                                    "callback, no MFMA and no tile prefetching");
        }
        if ((c.flags & fft1d_stage_out) &&
            (c.Mb != M || !packed_columns(M, n_out, c.ostride) || c.store_function)) {
            throw bad_configuration("Staged output needs packed columns, one M tile and no store "
                                    "callback");
        }
        if (!c.local_offsets()) {
            throw bad_configuration("Staged tiles need 32-bit tile offsets");
        }
        if (c.lds_bytes() > info.local_memory_size) {
            throw bad_configuration("Work-group exceeds the local memory size");
        }
    }
    if (c.flags & fft1d_direct_matrix) {
        if (!c.local_offsets() || c.work_group_size() > wg_max) {
            throw bad_configuration("Matrix sums need 32-bit tile offsets and a work-group of "
                                    "whole waves");
        }
    }
    if ((c.flags & fft1d_adjoint) && cfg.type == transform_type::c2c) {
        throw bad_configuration("The adjoint variant applies to real transforms only");
    }
    c.inplace_unsupported = cfg.type != transform_type::c2c && (c.Mb < M || inplace_refused);
    return c;
}

} // namespace bbfft

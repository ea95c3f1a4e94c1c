// The rule of lucida_amd/csrc/film_groups.hpp over given and random film sizes.
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#include "film_groups.hpp"

struct Film {
    uint32_t width, height;
};

static void expect(bool ok, const char* what) {
    if (ok) return;
    std::printf("failed: %s\n", what);
    std::exit(1);
}

static std::vector<size_t> groups(const std::vector<Film>& films) {
    std::vector<const Film*> in;
    for (const Film& f : films) in.push_back(&f);
    std::vector<size_t> out;
    for (size_t at = 0; at < in.size(); at += out.back()) {
        out.push_back(lucida::films_together(in.data() + at, in.size() - at, 16));
        expect(out.back() >= 1 && out.back() <= 16, "a launch takes one film at least and sixteen at most");
        uint64_t w = 0, h = 0, pixels = 0;
        for (size_t k = at; k < at + out.back(); ++k) {
            w = std::max<uint64_t>(w, in[k]->width);
            h = std::max<uint64_t>(h, in[k]->height);
            pixels += (uint64_t)in[k]->width * in[k]->height;
        }
        expect(out.back() == 1 || (double)out.back() * w * h <= 2.0 * pixels + lucida::EMPTY_PIXELS, "a bounded grid");
    }
    return out;
}

int main() {
    using V = std::vector<size_t>;
    expect(groups(std::vector<Film>(8, {256, 256})) == V{8}, "crops of one size together");
    expect(groups(std::vector<Film>(20, {256, 24})) == (V{16, 4}), "sixteen a launch");
    expect(groups({{256, 24}, {128, 8}, {130, 40}, {300, 9}}) == V{4}, "small films of any shape together");
    expect(groups({{1, 1}}) == V{1}, "one film");
    expect(groups({{131072, 16}, {128, 16384}}) == (V{1, 1}), "a wide and a tall film apart");
    expect(groups({{131072, 16}, {131072, 20}, {128, 16384}}) == (V{2, 1}), "the like-shaped ones of them together");
    expect(groups({{4294967295u, 1}, {1, 4294967295u}}) == (V{1, 1}), "no overflow");
    std::mt19937 rng(1);
    for (int rep = 0; rep < 2000; ++rep) {
        std::vector<Film> films(1 + rng() % 40);
        for (Film& f : films) f = {1u + (rng() >> (rng() % 20 + 12)), 1u + (rng() >> (rng() % 20 + 12))};
        groups(films);
    }
    std::printf("ok\n");
    return 0;
}

// Prints what the single-image tile rule picks: one line "shape blue cols count
// variant" on stdin, one line "threads two_lines" on stdout (256 CUs).  A length
// and an axis in place of the shape, "n <length> <cols>", print its shape, "one
// <width> <height>" whether the image runs in one launch.
#include <cstdint>
#include <iostream>
#include <string>

// from math_amd/csrc/host/runtime.hpp, without the HIP headers it needs
namespace mdft {
struct AxisTile {
    int threads;
    bool x2;
};
AxisTile axis_tile(int shape, bool blue, bool cols, int count, int variant, int cu_count);
int line_shape(long long n, bool cols);
struct LineFit {
    int tpl = 1;
    int conv = 0;
};
LineFit line_fit(long long n, bool cols);
bool one_launch(const LineFit& row, const LineFit& col, int w, int h);
}  // namespace mdft

int main()
{
    std::string first;
    while (std::cin >> first) {
        if (first == "n") {
            long long n;
            bool cols;
            std::cin >> n >> cols;
            std::cout << mdft::line_shape(n, cols) << "\n";
            continue;
        }
        if (first == "one") {
            int w, h;
            std::cin >> w >> h;
            std::cout << mdft::one_launch(mdft::line_fit(w, false), mdft::line_fit(h, true), w, h) << "\n";
            continue;
        }
        bool blue, cols;
        int count, variant;
        std::cin >> blue >> cols >> count >> variant;
        const mdft::AxisTile t = mdft::axis_tile(std::stoi(first), blue, cols, count, variant, 256);
        std::cout << t.threads << " " << t.x2 << "\n";
    }
    return 0;
}

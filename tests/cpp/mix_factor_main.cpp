// Prints the radices of every length from 17 to 8192 points that the mixed-radix kernel takes in one pass:
// "length radix radix ...".  Links the library's own mix_factor.
#include <cstdio>
#include <vector>

namespace ifft {
bool mix_factor(int N, int max_threads, std::vector<int> &radices, int &threads, double *cost_out, int min_stages);
}

int main()
{
    for (int n = 17; n <= 8192; ++n) {
        int m = n;
        for (int p : {2, 3, 5, 7, 11, 13})
            while (m % p == 0) m /= p;
        if (m != 1 || (n >= 64 && (n & (n - 1)) == 0)) continue;   // powers of two have their own kernel
        std::vector<int> r;
        int nt;
        double cost;
        if (!ifft::mix_factor(n, 512, r, nt, &cost, 2)) continue;
        std::printf("%d", n);
        for (int x : r) std::printf(" %d", x);
        std::printf("\n");
    }
    return 0;
}

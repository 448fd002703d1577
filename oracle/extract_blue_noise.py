"""Extract the 64x64 blue-noise threshold matrix (Pixman's generated matrix)
into a C header for the oracle build: from the reference's
src/internal/blue_noise.zig, or from the library's blue_noise_64x64.inc where
the reference's source is absent."""
import re
import sys

src, dst = sys.argv[1], sys.argv[2]
text = open(src).read()
if "= .{" in text:
    body = text[text.index("= .{") + 4: text.rindex("};")]
else:
    body = "\n".join(ln for ln in text.splitlines() if not ln.startswith("//"))
vals = [int(v) for v in re.findall(r"\d+", body)]
assert len(vals) == 4096, len(vals)
with open(dst, "w") as f:
    f.write("/* generated by oracle/extract_blue_noise.py; Pixman blue-noise\n"
            " * matrix (see the reference's LICENSE for the Pixman licence) */\n")
    f.write("static const unsigned short zo_blue_noise_64x64[4096] = {\n")
    for i in range(0, 4096, 16):
        f.write("  " + ", ".join(str(v) for v in vals[i:i + 16]) + ",\n")
    f.write("};\n")
